// cx_few.h — one fp8 expert over a few tokens (one decode batch), as two
// launches in which a wave's loads are one round trip and every CU streams.
// Semantics: RunFusedUpGateReferenceV2 / RunDownReferenceV2
// (expert_node_v2/backend/expert_reference_v2.cc:11-144), dequantise-then-fp32,
// h kept to 16 significant bits (bf16 hi + lo).
//
// At this size HBM is not the bound but each wave's chain of loads, and a grid
// of 16-row tiles leaves half of the CUs idle:
//  * gate/up (k_gu_few): a workgroup's 16 MFMA rows are 8 gate rows and the 8 up
//    rows of the same outputs, so inter / 8 workgroups (256 at 2048) each finish
//    their h; K is split over the 8 waves.  MFMA step j of a 128-column block
//    covers k = 32 j + 8 g in lane group g, so that every load instruction, of
//    weights (8 B a lane) and of x (16 B a lane), reads runs of 64 bytes or more.
//  * h goes to memory in the order in which the down projection's MFMA fragments
//    read it: per 16-token tile and 128 columns, [plane][step][lane][8], k = 32 g
//    + 8 j, one contiguous 1 KB load each.
//  * down (k_dn_few): 32 rows per workgroup, K split over its 4 waves.
// One expert of 7168 x 2048, us a launch, before (16-row tiles over the full K,
// or above 16 tokens the ping-pong GEMM) and now: gate/up at 5 / 13 / 16 / 32 / 64
// tokens 8.8 -> 8.1, 10.3 -> 9.3, 10.7 -> 9.5, 27 -> 13.4, 27 -> 20; down 11.7 ->
// 6.0, 16.8 -> 6.0, 19.2 -> 6.0, 13.2 -> 7.6, 13.3 -> 9.7.
#pragma once

#include "cx_down.h"
#include "cx_grouped.h"

namespace cx {

constexpr int kFewGuRows = 8;    // outputs per gate/up workgroup
constexpr int kFewDnRows = 32;
constexpr int kFewDnWaves = 4;

// Gate/up: NKB blocks per wave, KSA waves with work, NT column tiles, D blocks of
// x in flight.  x is loaded as whole rows of a block (4 tokens x 256 B an
// instruction, none for rows past the last token) and handed to the MFMA
// fragments through the wave's own LDS, chunk q of token t at q ^ t: loaded
// straight into fragment order, 16 tokens x 64 B an instruction, one expert's
// gate/up took 8.6 / 12.7 / 29 us at 1 / 16 / 64 tokens.

template <int NKB, int KSA, int NT, int D, bool F16>
__device__ __forceinline__ void few_gate_up(const ExpertLaunch& L, unsigned char* lds) {
    typedef Mma<F16> M;
    const cx_expert_desc& e = L.single;
    const int H = L.hidden, nkbi = L.inter / kKB;
    const int wave = wave_id(), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int r0 = blockIdx.x * kFewGuRows, np = L.n_tokens;
    unsigned char* own = lds + wave * (NT * 4096);  // x of a block, then the wave's partial tiles
    if (wave < KSA) {
        const int kb0 = wave * NKB;
        const int gl = __builtin_amdgcn_readfirstlane(e.gu_layout);
        const uint8_t* wp = (c < 8 ? e.w_gate : e.w_up) + gu_elem_off(gl, H, r0 + (c & 7), kb0 * kKB) + 8 * g;
        const int kw = gu_kstep(gl), jw = gl == CX_LAYOUT_TILE16 ? 512 : 32;  // bytes between blocks, steps
        // this lane's x pieces: token 4 i + lane / 16, chunk lane % 16; a token past
        // the last reads zero (bounded buffer), a whole instruction of them is left out
        const __amdgpu_buffer_rsrc_t xres =
            make_rsrc(L.x, (uint32_t)np * (uint32_t)H * 2);
        const uint32_t xo = ((uint32_t)g * (uint32_t)H + kb0 * kKB + 8 * c) * 2;
        unsigned char* xw = own + g * 256;
        const float* sg = e.s_gate + (size_t)__builtin_amdgcn_readfirstlane(r0 / e.gate_rb) * (H / kKB) + kb0;
        const float* su = e.s_up + (size_t)__builtin_amdgcn_readfirstlane(r0 / e.up_rb) * (H / kKB) + kb0;
        u32x2 w[NKB][4];
        u32x4 xr[D][4 * NT];
        auto load_x = [&](int k) {
#pragma unroll
            for (int i = 0; i < 4 * NT; ++i)
                if (4 * i < np) xr[k % D][i] = bld16(xres, xo + (uint32_t)i * 8 * H + k * kKB * 2);
        };
#pragma unroll
        for (int k = 0; k < NKB; ++k) {
#pragma unroll
            for (int j = 0; j < 4; ++j) w[k][j] = ld8(wp + (size_t)k * kw + j * jw);
            if (k < D) load_x(k);
            __builtin_amdgcn_sched_barrier(0);
        }
        float scg[NKB], scu[NKB];
#pragma unroll
        for (int k = 0; k < NKB; ++k) {
            scg[k] = ldsc(sg + k);
            scu[k] = ldsc(su + k);
        }
        f32x4 acc[NT];
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt] = zero;
#pragma unroll
        for (int k = 0; k < NKB; ++k) {
            const float sc = g < 2 ? scg[k] : scu[k];  // rows 4 g ..: gate below 8, up from 8
            // (a wave's LDS accesses execute in order: no wait between them)
#pragma unroll
            for (int i = 0; i < 4 * NT; ++i)
                if (4 * i < np)
                    *reinterpret_cast<u32x4*>(xw + i * 1024 + 16 * (c ^ ((4 * i + g) & 15))) = xr[k % D][i];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
                f32x4 t = zero;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const u32x4 b = *reinterpret_cast<const u32x4*>(own + tt * 4096 + c * 256 + 16 * ((4 * j + g) ^ c));
                    t = M::mma(M::cvt(w[k][j][0], w[k][j][1]), M::bits(b), t);
                }
                acc[tt] += sc * t;
            }
            __builtin_amdgcn_sched_barrier(0);
            if (k + D < NKB) load_x(k + D);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) reinterpret_cast<f32x4*>(own)[tt * 64 + lane] = acc[tt];
    }
    const f32x4* red = reinterpret_cast<const f32x4*>(lds);  // wave v's tile tt at v * NT * 256 + tt * 64
    __syncthreads();
    for (int tt = wave; tt < NT; tt += kFewGuWaves) {
        f32x4 s = red[tt * 64 + lane];
#pragma unroll
        for (int v = 1; v < KSA; ++v) s += red[v * NT * 256 + tt * 64 + lane];
        // lanes 0..31 hold gate rows 4 g .., lanes 32..63 the up rows of the same
        uint32_t hi[4], lo[4];
        float hv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float gate = s[i], up = __shfl(s[i], (lane + 32) & 63, 64);
            const float h = (gate / (1.0f + expf(-gate))) * up;
            hv[i] = h;
            hi[i] = bf16_rne(h);
            lo[i] = bf16_rne(h - __uint_as_float(hi[i] << 16));
        }
        if (lane < 32 && tt * kTileTok + c < np) {
            const int r = r0 + 4 * g;  // k of the down projection: block r / 128, group r / 32 % 4, step r / 8 % 4
            const size_t o = ((size_t)tt * nkbi + (r >> 7)) * kFewHBlk + ((r >> 3) & 3) * 1024 +
                             (((r >> 5) & 3) * 16 + c) * 16 + (r & 4) * 2;
            unsigned char* hp = reinterpret_cast<unsigned char*>(L.h_hi) + o;
            *reinterpret_cast<uint2*>(hp) = uint2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
            *reinterpret_cast<uint2*>(hp + kFewHBlk / 2) = uint2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
            if (L.h_f32 != nullptr)
                *reinterpret_cast<float4*>(L.h_f32 + (size_t)(tt * kTileTok + c) * L.inter + r) = float4{hv[0], hv[1], hv[2], hv[3]};
        }
    }
}

// Down: NKB blocks per wave, NT column tiles, D blocks of h in flight.
template <int NKB, int NT, int D>
__device__ __forceinline__ void few_down(const ExpertLaunch& L, unsigned char* lds) {
    const cx_expert_desc& e = L.single;
    const int H = L.hidden, I = L.inter;
    const int wave = wave_id(), lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int r0 = blockIdx.x * kFewDnRows, np = L.n_tokens;
    const int kb0 = wave * NKB;
    f32x4* red = reinterpret_cast<f32x4*>(lds);  // [kFewDnWaves][2 NT][64]
    const uint8_t* wp = e.w_down + (size_t)(r0 + c) * I + kb0 * kKB + 32 * g;
    const unsigned char* hp = reinterpret_cast<const unsigned char*>(L.h_hi) + kb0 * kFewHBlk + lane * 16;
    const size_t htile = (size_t)(I / kKB) * kFewHBlk;
    u32x4 w[2][NKB][2];
    u32x4 hb[D][NT][8];
    auto load_h = [&](int k) {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
            for (int j = 0; j < 8; ++j) hb[k % D][tt][j] = ld16(hp + tt * htile + k * kFewHBlk + j * 1024);
    };
#pragma unroll
    for (int k = 0; k < NKB; ++k) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            w[m][k][0] = ld16(wp + (size_t)m * kTileRows * I + k * kKB);
            w[m][k][1] = ld16(wp + (size_t)m * kTileRows * I + k * kKB + 16);
        }
        if (k < D) load_h(k);
        __builtin_amdgcn_sched_barrier(0);
    }
    float sd[2][NKB];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const float* sp = e.s_down + (size_t)__builtin_amdgcn_readfirstlane((r0 + m * kTileRows) / e.down_rb) * (I / kKB) + kb0;
#pragma unroll
        for (int k = 0; k < NKB; ++k) sd[m][k] = ldsc(sp + k);
    }
    f32x4 acc[2][NT];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[m][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NKB; ++k) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) acc[m][tt] += sd[m][k] * down_step(w[m][k], hb[k % D][tt]);
        __builtin_amdgcn_sched_barrier(0);
        if (k + D < NKB) load_h(k + D);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) red[((wave * 2 + m) * NT + tt) * 64 + lane] = acc[m][tt];
    __syncthreads();
    for (int i = wave; i < 2 * NT; i += kFewDnWaves) {
        const int m = i / NT, tt = i % NT;
        f32x4 s = red[i * 64 + lane];
#pragma unroll
        for (int v = 1; v < kFewDnWaves; ++v) s += red[(v * 2 * NT + i) * 64 + lane];
        const int q = tt * kTileTok + c;
        if (q < np) store_out4(L.y, L.y_f32, (size_t)q * H + r0 + m * kTileRows + 4 * g, s, L.out_dtype);
    }
}

}  // namespace cx
