// cx_pp.h — the grouped fp8 expert MLP as two GEMM kernels on a ring of LDS stages
// whose two waves per SIMD alternate between loading and multiplying (ping-pong),
// for items of up to 128 pairs: prefill chunks with many tokens per expert
// (big_min_pairs), and one expert over more than 64 tokens (more than 16 at widths
// without few-token kernels).
// Semantics: RunFusedUpGateReferenceV2 / RunDownReferenceV2
// (expert_node_v2/backend/expert_reference_v2.cc:11-144) per expert,
// dequantise-then-fp32, h kept to 16 significant bits (bf16 hi + lo).
#pragma once

#include <type_traits>

#include "cx_gate_up.h"
#include "cx_grouped.h"

namespace cx {

constexpr int kPpK = 64;        // k of half a 128-column scale block
constexpr int kPpA = 16384;     // weight bytes of a half block: 16 tiles x 16 rows x 64 k
constexpr int kPpTile = 2048;   // activation bytes of a 16-pair column tile and plane in a half block
constexpr int kPpMaxTiles = kBigPairs / kTileTok;

// Weight tiles per wave.  The down projection of more than four column tiles
// splits the columns over the two waves of a SIMD (see pp_core), which computes
// an even count.
constexpr int pp_wtiles(int nt, int planes) { return planes == 2 && nt > 4 ? 4 : 2; }
constexpr int pp_tiles(int nt, int planes) { return pp_wtiles(nt, planes) == 4 ? (nt + 1) / 2 * 2 : nt; }
// Half blocks per stage: items of up to four column tiles take gate/up stages
// of a whole 128-column block, so that a step still multiplies enough.
constexpr int pp_halves(int nt, int planes) { return planes == 1 && nt <= 4 ? 2 : 1; }
constexpr int pp_stage(int nt, int planes) { return pp_halves(nt, planes) * (kPpA + nt * planes * kPpTile); }
// Stages in the ring.
constexpr int pp_ring(int nt, int planes) {
    const int r = kPpLds / pp_stage(nt, planes);
    return r > 7 ? 7 : r;
}

// Loads per half block (or plane) and wave: the activations of four column
// tiles as one 16-byte-per-lane load, a leftover tile as one 4-byte-per-lane
// load, so that every wave issues the same number.
constexpr int pp_bloads(int nt) { return nt / 4 + nt % 4; }

__device__ __forceinline__ uint32_t pp_lds_addr(const unsigned char* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)p;
}
// Fragment reads as asm: as plain loads the compiler cannot tell which stage a
// pending global->LDS DMA writes and drains the ring (vmcnt(0)) before them.
// Every output is an operand of pp_lds_wait, so it stays live and unread until
// the read has landed.
template <int OFF>
__device__ __forceinline__ void pp_read(u32x4& v, uint32_t base) {
    static_assert(OFF >= 0 && OFF < 65536 && OFF % 16 == 0, "ds_read offset field");
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(OFF));
}
// f(integral_constant 0), ..., f(integral_constant N - 1)
template <int N, int I = 0, class F>
__device__ __forceinline__ void pp_steps(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        pp_steps<N, I + 1>(f);
    }
}
__device__ __forceinline__ void pp_pin(u32x4& v) { asm volatile("" : "+v"(v)); }
// LDS reads return in order: with N younger ones in flight, `a` has landed.
template <int N, int M>
__device__ __forceinline__ void pp_lds_wait(u32x4 (&v)[M]) {
    static_assert(N < 16, "lgkmcnt range");
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v[0]) : "i"(N));
#pragma unroll
    for (int i = 1; i < M; ++i) pp_pin(v[i]);
}

__device__ __forceinline__ void pp_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Where a lane's activation loads come from: its pairs' rows (byte pointers at
// the lane's place in the row) for each of the wave's loads of a stage.
template <int NT>
struct PpSrc {
    static constexpr int N = pp_bloads(NT);
    const unsigned char* p[N];
};

// Activation rows of a stage: 128 B (64 values) per pair, 16-byte chunk q of
// pair t at chunk q ^ (t & 7) ^ ((t >> 3) & 1) (measured free of bank conflicts
// for the fragment reads).  Load m < nt / 4 covers pairs 64 m + 8 wave + lane / 8;
// a leftover tile's load covers its pairs 2 wave + lane / 32.  row(q): the
// first byte of pair q's row.
template <int NT, class Row>
__device__ __forceinline__ void pp_sources(PpSrc<NT>& s, int wave, int lane, Row row) {
#pragma unroll
    for (int m = 0; m < PpSrc<NT>::N; ++m) {
        if (m < NT / 4) {
            const int t = 64 * m + 8 * wave + (lane >> 3);
            s.p[m] = row(t) + 16 * ((lane & 7) ^ (t & 7) ^ ((t >> 3) & 1));
        } else {
            const int t = 16 * (4 * (NT / 4) + m - NT / 4) + 2 * wave + (lane >> 5);
            const int d = lane & 31;
            s.p[m] = row(t) + 16 * ((d >> 2) ^ (t & 7) ^ ((t >> 3) & 1)) + 4 * (d & 3);
        }
    }
}

// Weights of a workgroup's 16 tiles of 16 rows.  A wave loads two 1 KB pieces
// per half block: lane pointers p0, p1, and the distances of the pieces.
//  * gate/up (LINES = false): the pieces are two tiles' half blocks, each lane's
//    16 bytes where its MFMA fragments read them; stage s at + (s / 2) * kw + (s % 2) * hw.
//  * down (LINES = true, row-major weights): a half block's worth of whole
//    128-byte row lines: stage 2 kb carries half of the wave's tiles for all 128
//    columns of block kb, stage 2 kb - 1 the other half (p0 / p1: rows 0..7 /
//    8..15 of a tile of stage -1; + hw: of stage 0; kw between blocks).  Read as
//    64-byte halves of lines, one expert's down over 128 tokens took 20.1
//    instead of 14.9 us.
struct PpW {
    const uint8_t* p0;
    const uint8_t* p1;
    int kw, hw;
};

// The GEMM of one workgroup: acc[m][tt] = sum over k of the wave's weight tile m
// times its column tile tt, the 128-column blocks scaled by sc[m][block] (wave-
// uniform).  src + plane * dplane: the planes' activations.
//
// MT = 2: wave w has tiles 2 w, 2 w + 1 and all columns.  MT = 4: waves w and
// w + 4 share tiles 4 (w % 4) .. + 3 and take half of the columns each: fewer LDS
// reads per product (20 instead of 34 KB per 64 MFMAs) for twice the weight
// conversions.  Measured at 128 pairs per item, 4096 tokens of one expert: down
// 206 us with 4 and 225 with 2 tiles per wave, gate/up 219 and 201.
//
// Stages go through a ring of LDS buffers by global->LDS DMA, RING - 1 ahead.
// Each step of a wave is L (read the step's fragments, convert its weights,
// issue a share of the loads, add the last block's scaled products) then C (its
// MFMAs).  The waves of a SIMD (w and w + 4) are kept half a step apart, so that
// one multiplies while the other loads: waves 4..7 pass the stage's barrier
// after their last L, waves 0..3 after their last C.  All reads of a stage so lie
// between two barriers; loads issued there go to the buffer of the stage before;
// a wave passes the barrier once its own loads of the next stage have landed.
template <int NT, int PL, int RING, bool F16, int MT, int NW>
__device__ __forceinline__ void pp_core(PpW w, PpSrc<NT> src, ptrdiff_t dplane, int nkb, const float* (&sc)[MT],
                                        unsigned char* lds, f32x4 (&acc)[MT][NW]) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass cannot parse the asm constraints
    typedef Mma<F16> M;
    typedef typename M::V V;
    constexpr bool LINES = PL == 2;
    constexpr int HS = pp_halves(NT, PL), HB = 2 / HS;  // half blocks per stage, stages per block
    constexpr int P = PL == 2 && NT > 4 ? 2 : 1;        // steps per stage
    constexpr int G = HS * PL * 2 / P;                  // (MFMA step, plane)s per step
    constexpr int NA = HS * 2 / P;                      // MFMA steps per step
    constexpr int NB = PpSrc<NT>::N, LPS = HS * (2 + PL * NB), STAGE = pp_stage(NT, PL);
    static_assert(MT * NW == 2 * NT && (MT == 2 || MT == 4), "tile shape");
    static_assert(NT >= 1 && NT <= kPpMaxTiles && (PL == 1 || PL == 2), "tile shape");
    static_assert(RING >= 3 && (RING - 1 + HB - 1) / HB <= kPpMinBlocks, "ring");
    const int wave = wave_id(), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const bool second = wave >= 4;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const uint32_t l0 = pp_lds_addr(lds);
    // where this wave's weight pieces go and where its tiles are read from
    const int adst = MT == 2 ? wave * 2048 : (wave & 3) * 4096 + (wave >> 2) * 2048;
    const uint32_t ab = l0 + (MT == 2 ? wave * 2048 : (wave & 3) * 4096);
    const int key = (c & 7) ^ ((c >> 3) & 1);
    uint32_t ard[2];  // LINES: by half block; else by lane order
    ard[0] = ab + (LINES ? c * 128 + 16 * (g ^ key) : lane * 16);
    ard[1] = ab + (LINES ? c * 128 + 16 * ((4 + g) ^ key) : lane * 16);
    uint32_t brd[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        brd[j] = l0 + HS * kPpA + (MT == 4 && second ? NW * kPpTile : 0) + c * 128 + 16 * ((2 * g + j) ^ key);
    int islot = 0, rslot = 0;  // byte offsets of the slots issued / read next
    // load i of the stage to issue (weights, then the planes' activations)
    auto issue_weights = [&](int i, int slot) {
        const int hf = i >> 1, m = i & 1;
        __builtin_amdgcn_global_load_lds((m == 0 ? w.p0 : w.p1) + hf * w.hw, lds + slot + hf * kPpA + adst + m * 1024, 16, 0, 0);
    };
    auto issue_load = [&](int i) {
        if (i < 2 * HS) {
            issue_weights(i, islot);
        } else {
            const int k = (i - 2 * HS) / NB, m = (i - 2 * HS) % NB;  // half (PL = 1) or plane
            const unsigned char* sp = src.p[m] + (PL == 2 ? k * dplane : (ptrdiff_t)(k * 2 * kPpK));
            unsigned char* db = lds + islot + HS * kPpA + k * NT * kPpTile;
            if (m < NT / 4) __builtin_amdgcn_global_load_lds(sp, db + m * 8192 + wave * 1024, 16, 0, 0);
            else __builtin_amdgcn_global_load_lds(sp, db + (4 * (NT / 4) + m - NT / 4) * kPpTile + wave * 256, 4, 0, 0);
        }
    };
    int ib = 0;  // LINES: block of the weights issued next
    auto next_weights = [&](bool odd) {  // `odd`: the stage just issued (compile-time)
        int da;
        if (HS == 2) da = w.kw;
        else if (!LINES) da = odd ? w.kw - w.hw : w.hw;
        else da = odd ? w.hw : (ib < nkb - 1 ? w.kw : 0) - w.hw;  // past the last block: its own weights again
        if (LINES && !odd) ++ib;
        w.p0 += da;
        w.p1 += da;
    };
    auto issue_next = [&](bool odd) {
        next_weights(odd);
#pragma unroll
        for (int m = 0; m < NB; ++m) src.p[m] += HS * 2 * kPpK;
        islot = islot == (RING - 1) * STAGE ? 0 : islot + STAGE;
    };
    if constexpr (LINES) {  // stage -1: the first tiles of block 0, through the last slot
        issue_weights(0, (RING - 1) * STAGE);
        issue_weights(1, (RING - 1) * STAGE);
        next_weights(true);
    }
#pragma unroll
    for (int s = 0; s < RING - 1; ++s) {
#pragma unroll
        for (int i = 0; i < LPS; ++i) issue_load(i);
        issue_next(s & 1);
    }
    // raw weights: LINES: [tile][half block]; else [half block of the stage][tile]
    constexpr int NRAW = LINES ? 2 * MT : HS * MT;
    u32x4 aw[NRAW];
    u32x4 an[LINES ? MT : 1];  // LINES: the next block's first tiles
    vm_wait<(RING - 2) * LPS>();
    pp_barrier();
    if constexpr (LINES) {
        pp_steps<MT>([&](auto i) { pp_read<(i.value >> 1) * 2048>(an[i.value], ard[i.value & 1] + (RING - 1) * STAGE); });
        pp_lds_wait<0>(an);
        pp_barrier();
    }

    f32x4 part[MT][NW];
    // the multiplied block's scales, and the next one's, loaded a block ahead
    float s0[MT], sn[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        s0[m] = 0.f;
        sn[m] = ldsc(sc[m]);
    }
    auto scaled_add = [&](int i) {  // accumulator i
        const int m = i % MT, tt = i / MT;
        acc[m][tt] += s0[m] * part[m][tt];
        asm volatile("" : "+v"(acc[m][tt]));
    };
    V a[MT][NA];
    // weight fragment i of a step of stage h: tile i % MT, MFMA step i / MT (of the stage: + ph)
    auto convert = [&](int i, int h, int ph) {
        const int m = i % MT, j = P == 2 ? ph : i / MT;
        const u32x4 v = LINES ? aw[2 * m + h] : aw[(j >> 1) * MT + m];
        u32x4 t = __builtin_bit_cast(u32x4, M::cvt(v[2 * (j & 1)], v[2 * (j & 1) + 1]));
        asm volatile("" : "+v"(t));
        a[m][i / MT] = __builtin_bit_cast(V, t);
    };
    // block kb; tail (compile-time): blocks after it if it is one of the last
    // TB, whose stages issue and wait for what is left, else -1
    auto block = [&](int kb, auto tail) {
        constexpr int TJ = decltype(tail)::value;
        if constexpr (LINES) {
#pragma unroll
            for (int i = 0; i < MT; ++i) aw[i] = an[i];
        }
        pp_steps<HB * P>([&](auto step) {
            constexpr int h = step.value / P, ph = step.value % P;
            constexpr bool more = TJ < 0 || RING - 1 - HB - HB * TJ + h < 0;    // stage s + RING - 1 exists
            constexpr int left = HB * TJ + HB - 2 - h;                          // stages after s + 1
            constexpr int later = TJ < 0 || left > RING - 2 ? RING - 2 : left;  // of them in flight
            constexpr bool fresh = h == 0 && ph == 0;
            // L.  LDS reads, loads and VALU work queue in different units, so
            // they are interleaved.
            u32x4 bf[G * NW];  // [group][column tile]
            if (ph == 0) {
                if constexpr (!LINES) {
                    pp_steps<NRAW>([&](auto i) { pp_read<(i.value / MT) * kPpA + (i.value % MT) * 1024>(aw[i.value], ard[0] + rslot); });
                } else {
                    pp_steps<MT>([&](auto i) {  // tile pair MT / 2 + i / 2 of this block, or i / 2 of the next
                        pp_read<(i.value >> 1) * 2048>(h == 0 ? aw[MT + i.value] : an[i.value], ard[i.value & 1] + rslot);
                    });
                }
            }
            uint32_t gb[2];
            gb[0] = brd[P == 2 ? ph : 0] + rslot;
            gb[1] = (P == 2 ? brd[ph] + NT * kPpTile : brd[1]) + rslot;
            constexpr int NI = G * NW / 2;                       // read pairs
            constexpr int NF = (NI + 1) / 2;                     // pairs read before the weights are waited for
            constexpr int NR = NI > NF ? NI - NF : 1;
            constexpr int NCV = MT * NA;                         // weight fragments to convert
            constexpr int L0 = ph * LPS / P, LN = (ph + 1) * LPS / P - L0;  // this step's loads
            constexpr int ND = MT * NW;                          // accumulators
            pp_steps<NI>([&](auto ic) {
                constexpr int i = ic.value;
                pp_steps<2>([&](auto r) {
                    constexpr int f = 2 * i + r.value, gr = f / NW, tt = f % NW;
                    // group gr: P = 2: plane gr; else MFMA step gr % 2 of half gr / 2 (PL = 1), or
                    // plane gr % 2 of step gr / 2 (PL = 2)
                    constexpr int base = P == 2 ? gr : PL == 1 ? gr & 1 : gr >> 1;
                    constexpr int blk = P == 2 ? 0 : PL == 1 ? gr >> 1 : gr & 1;
                    pp_read<(blk * NT + tt) * kPpTile>(bf[f], gb[base]);
                });
                if (more) {
#pragma unroll
                    for (int q = i * LN / NI; q < (i + 1) * LN / NI; ++q) issue_load(L0 + q);
                }
                if (fresh) {
#pragma unroll
                    for (int q = i * ND / NI; q < (i + 1) * ND / NI; ++q) scaled_add(q);
                }
                if (i == NF - 1 && ph == 0) pp_lds_wait<2 * NF>(aw);
                if (i >= NF) {
#pragma unroll
                    for (int q = (i - NF) * NCV / NR; q < (i + 1 - NF) * NCV / NR; ++q) convert(q, h, ph);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if (NI == NF) {
#pragma unroll
                for (int q = 0; q < NCV; ++q) convert(q, h, ph);
            }
            if (more && ph == P - 1) issue_next((h + RING - 1) & 1);
            if constexpr (LINES && h == 1 && ph == 0) pp_lds_wait<0>(an);
            pp_lds_wait<0>(bf);
            if (ph == P - 1 && later >= 0) vm_wait<(later < 0 ? 0 : later) * LPS>();
            if (ph == P - 1 && second) pp_barrier();
            __builtin_amdgcn_sched_barrier(0);
            // C
            if (fresh) {
                const int kn = min(kb + 1, nkb - 1);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    s0[m] = sn[m];
                    asm volatile("" : "+s"(s0[m]));  // here, where no LDS read is in flight that the wait would cover
                }
#pragma unroll
                for (int m = 0; m < MT; ++m) sn[m] = ldsc(sc[m] + kn);
            }
            if (ph == P - 1) rslot = rslot == (RING - 1) * STAGE ? 0 : rslot + STAGE;
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int gr = 0; gr < G; ++gr)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int tt = 0; tt < NW; ++tt)
                        part[m][tt] = M::mma(a[m][P == 2 ? 0 : PL == 1 ? gr : gr >> 1], M::bits(bf[gr * NW + tt]),
                                             fresh && gr == 0 ? zero : part[m][tt]);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            if (ph == P - 1 && !second) pp_barrier();
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr int TB = (RING - 1 + HB - 1) / HB;  // blocks whose stages do not all issue a later one
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int tt = 0; tt < NW; ++tt) acc[m][tt] = part[m][tt] = zero;
    int kb = 0;
#pragma unroll 1
    for (; kb < nkb - TB; ++kb) block(kb, std::integral_constant<int, -1>{});
    pp_steps<TB>([&](auto t) { block(kb + t.value, std::integral_constant<int, TB - 1 - t.value>{}); });
#pragma unroll
    for (int i = 0; i < MT * NW; ++i) scaled_add(i);
#endif
}

// Workgroup b runs on XCD b % 8 (round-robin dispatch), one workgroup to a CU.
// The XCDs take the n logical tiles in turn, kPpChunk consecutive ones at a time
// (one per CU: row tiles of an item, which share its activations in that XCD's
// L2, and of the expert's next items, which share the weights), and an eighth
// each of what is left; -1 past the end.  Items differ in length, the shared
// expert's, all full, come last: with one contiguous eighth of the tiles per XCD
// a layer of 256 experts took 3240 us at 1511 and 4066 at 2500 tokens, with
// chunks 2948 and 3958 (16 or 64 tiles a chunk: within 1 % of 32).
constexpr int kPpChunk = 32;
__device__ __forceinline__ int pp_tile(int n) {
    const int b = blockIdx.x, x = b & 7, i = b >> 3;
    const int full = n / (8 * kPpChunk) * (8 * kPpChunk);
    if (b < full) return (i / kPpChunk * 8 + x) * kPpChunk + i % kPpChunk;
    const int per = (n - full + 7) >> 3, j = i - (full >> 3), t = full + x * per + j;
    return j < per && t < n ? t : -1;
}

// Logical tile -> (item, row tile): groups of kPpGroup consecutive items
// (an expert's items are consecutive in the plan) walk their row tiles
// together, so the workgroups that share a row tile's weights run side by
// side on one XCD and its L2 serves them one fetch.  false past the items.
constexpr int kPpGroup = 4;
__device__ __forceinline__ bool pp_item_tile(int t, int n_items, int n_rt, int* item, int* tile) {
    const int span = kPpGroup * n_rt;
    const int g = t / span, r = t - g * span;
    const int in_group = min(kPpGroup, n_items - g * kPpGroup);
    *tile = r / in_group;
    *item = g * kPpGroup + (r - *tile * in_group);
    return *tile < n_rt;
}

template <bool SINGLE>
__device__ __forceinline__ bool pp_unit(const ExpertLaunch& L, int n_rt, Unit* u, int* tile) {
    int n_items;
    if (SINGLE) {
        n_items = (L.n_tokens + L.item_cap - 1) / L.item_cap;
    } else {
        const PlanHdr hd = ld_uniform(L.plan.hdr);
        n_items = L.skip_shared ? hd.n_routed_items : hd.n_items;
    }
    const int t = pp_tile(n_items * n_rt);
    if (t < 0) return false;
    int item;
    if (!pp_item_tile(t, n_items, n_rt, &item, tile)) return false;
    return resolve_unit<SINGLE>(L, item, SINGLE ? L.item_cap : kBigPairs, u);
}

// ---------------------------------------------------------------------------
// gate/up: a wave's tiles are 16 gate rows and the up rows of the same
template <int NT, bool F16, bool SINGLE>
__device__ __forceinline__ void pp_gate_up_item(const ExpertLaunch& L, const Unit& u, int tile, unsigned char* lds) {
    const int H = u.e.hidden, I = u.e.inter, nkb = H / kKB;
    const int wave = wave_id(), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int r0 = tile * kPpRowsGu + wave * kTileRows;
    const int gl = __builtin_amdgcn_readfirstlane(u.e.gu_layout);
    const bool tiled = gl == CX_LAYOUT_TILE16;
    const size_t ao = gu_elem_off(gl, H, r0 + c, 16 * g);
    const PpW w{u.e.w_gate + ao, u.e.w_up + ao, tiled ? 2048 : kKB, tiled ? 1024 : kPpK};
    PpSrc<NT> src;
    pp_sources<NT>(src, wave, lane, [&](int t) {
        const int q = u.pb + min(t, u.np - 1);
        const int tok = SINGLE ? q : ldi(L.plan.pair_token + q);
        return static_cast<const unsigned char*>(L.x) + (size_t)tok * H * 2;
    });
    const float* scales[2] = {
        u.e.s_gate + (size_t)__builtin_amdgcn_readfirstlane(r0 / u.e.gate_rb) * nkb,
        u.e.s_up + (size_t)__builtin_amdgcn_readfirstlane(r0 / u.e.up_rb) * nkb};
    f32x4 acc[2][NT];
    pp_core<NT, 1, pp_ring(NT, 1), F16, 2, NT>(w, src, 0, nkb, scales, lds, acc);
    // SiLU(gate) * up -> h as bf16 hi + lo, per pair
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
        const int q = tt * kTileTok + c;
        if (q >= u.np) continue;
        const size_t o = (size_t)(u.pb + q) * I + r0 + 4 * g;
        uint32_t hi[4], lo[4];
        float hv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float gate = acc[0][tt][i], up = acc[1][tt][i];
            const float hh = (gate / (1.0f + expf(-gate))) * up;
            hv[i] = hh;
            hi[i] = bf16_rne(hv[i]);
            lo[i] = bf16_rne(hv[i] - __uint_as_float(hi[i] << 16));
        }
        *reinterpret_cast<uint2*>(L.h_hi + o) = uint2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
        *reinterpret_cast<uint2*>(L.h_lo + o) = uint2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
        if (L.h_f32 != nullptr) *reinterpret_cast<float4*>(L.h_f32 + o) = float4{hv[0], hv[1], hv[2], hv[3]};
    }
}

// ---------------------------------------------------------------------------
// down: h as hi + lo planes, both multiplied with the same converted weights
template <int NT, bool SINGLE>
__device__ __forceinline__ void pp_down_item(const ExpertLaunch& L, const Unit& u, int tile, unsigned char* lds) {
    constexpr int MT = pp_wtiles(NT, 2), NW = 2 * NT / MT;
    const int H = u.e.hidden, I = u.e.inter, nkb = I / kKB;
    const int wave = wave_id(), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int r0 = tile * kPpRowsDn + (MT == 2 ? wave : wave & 3) * MT * kTileRows;
    // pieces: rows 0..7 and 8..15 of a tile, whole 128-byte lines with the chunks
    // swizzled by row; stage -1 carries tile 0 (MT = 4: 0 and 1), stage 0 the rest
    PpW w;
    {
        const int row = lane >> 3;
        const uint8_t* base = u.e.w_down + (size_t)(r0 + (MT == 4 && wave >= 4 ? kTileRows : 0) + row) * I;
        w.p0 = base + 16 * ((lane & 7) ^ row);
        w.p1 = base + (size_t)8 * I + 16 * ((lane & 7) ^ row ^ 1);
    }
    w.kw = kKB;
    w.hw = MT / 2 * kTileRows * I;
    PpSrc<NT> src;
    pp_sources<NT>(src, wave, lane, [&](int t) {
        return reinterpret_cast<const unsigned char*>(L.h_hi + (size_t)(u.pb + min(t, u.np - 1)) * I);
    });
    const ptrdiff_t dplane = reinterpret_cast<const unsigned char*>(L.h_lo) - reinterpret_cast<const unsigned char*>(L.h_hi);
    const float* scales[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
        scales[m] = u.e.s_down + (size_t)__builtin_amdgcn_readfirstlane((r0 + m * kTileRows) / u.e.down_rb) * nkb;
    f32x4 acc[MT][NW];
    pp_core<NT, 2, pp_ring(NT, 2), false, MT, NW>(w, src, dplane, nkb, scales, lds, acc);
    const int c0 = MT == 4 && wave >= 4 ? NW : 0;
#pragma unroll
    for (int tt = 0; tt < NW; ++tt) {
        const int q = (c0 + tt) * kTileTok + c;
        if (q >= u.np) continue;
        const size_t o = (size_t)(u.pb + q) * H + r0 + 4 * g;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const f32x4 v = acc[m][tt];
            if (SINGLE) store_out4(L.y, L.y_f32, o + m * kTileRows, v, L.out_dtype);
            // read once, by the combine launch: streamed stores
            else __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(L.y_part + o + m * kTileRows));
        }
    }
}

// An item takes the code of its own count of column tiles (a uniform branch).
template <int PL, int NT = 1, class F>
__device__ __forceinline__ void pp_pick(int nt, F f) {
    if constexpr (NT <= kPpMaxTiles) {
        if (nt <= NT) f(std::integral_constant<int, NT>{});
        else pp_pick<PL, pp_tiles(NT + 1, PL)>(nt, f);
    }
}

template <bool F16, bool SINGLE>
__device__ __forceinline__ void pp_gate_up(const ExpertLaunch& L, unsigned char* lds) {
    Unit u;
    int tile;
    if (!pp_unit<SINGLE>(L, L.inter / kPpRowsGu, &u, &tile)) return;
    pp_pick<1>((u.np + kTileTok - 1) / kTileTok, [&](auto nt) { pp_gate_up_item<nt.value, F16, SINGLE>(L, u, tile, lds); });
}

template <bool SINGLE>
__device__ __forceinline__ void pp_down(const ExpertLaunch& L, unsigned char* lds) {
    Unit u;
    int tile;
    if (!pp_unit<SINGLE>(L, L.hidden / kPpRowsDn, &u, &tile)) return;
    pp_pick<2>((u.np + kTileTok - 1) / kTileTok, [&](auto nt) { pp_down_item<nt.value, SINGLE>(L, u, tile, lds); });
}

}  // namespace cx
