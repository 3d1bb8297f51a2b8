// cx_few.hip — kernels and launchers of one expert over a few tokens (cx_few.h).
#include "cx_few.h"

namespace cx {
namespace {

template <int NKB, int KSA, int NT, int D, bool F16>
__global__ __launch_bounds__(64 * kFewGuWaves) __attribute__((amdgpu_waves_per_eu(2))) void k_gu_few(ExpertLaunch L) {
    extern __shared__ __attribute__((aligned(16))) unsigned char few_lds[];
    few_gate_up<NKB, KSA, NT, D, F16>(L, few_lds);
}

template <int NKB, int NT, int D>
__global__ __launch_bounds__(64 * kFewDnWaves) __attribute__((amdgpu_waves_per_eu(1))) void k_dn_few(ExpertLaunch L) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[kFewDnWaves * 2 * NT * 1024];
    few_down<NKB, NT, D>(L, lds);
}

template <int NKB, int KSA, int NT, bool F16>
void go_gu(const ExpertLaunch& L, hipStream_t s) {
    // blocks of x in flight within 256 registers (two waves per SIMD)
    constexpr int D = NT == 1 ? NKB : NT == 2 ? 4 : 2;
    const dim3 grid(L.inter / kFewGuRows);
    cx_launch((k_gu_few<NKB, KSA, NT, (D < NKB ? D : NKB), F16>), grid, dim3(64 * kFewGuWaves), few_gu_lds(NT), s, L);
}

template <int NT, bool F16>
void pick_gu(const ExpertLaunch& L, hipStream_t s) {
    switch (L.hidden / kKB) {
        case 56: go_gu<7, 8, NT, F16>(L, s); break;
        case 8: go_gu<1, 8, NT, F16>(L, s); break;
        default: go_gu<1, 4, NT, F16>(L, s); break;
    }
}

template <int NKB, int NT>
void go_dn(const ExpertLaunch& L, hipStream_t s) {
    constexpr int D = NT <= 2 ? NKB : 2;  // blocks of h in flight (one wave per SIMD)
    const dim3 grid(L.hidden / kFewDnRows);
    cx_launch((k_dn_few<NKB, NT, (D < NKB ? D : NKB)>), grid, dim3(64 * kFewDnWaves), 0, s, L);
}

}  // namespace

hipError_t launch_gate_up_few(const ExpertLaunch& L, hipStream_t s) {
    if (L.table != nullptr || !few_ok(L.hidden, L.inter, L.n_tokens, L.max_lds)) return hipErrorInvalidValue;
    const bool f16 = L.in_dtype == CX_DTYPE_FP16;
    switch (few_tiles(L.n_tokens)) {
        case 1: f16 ? pick_gu<1, true>(L, s) : pick_gu<1, false>(L, s); break;
        case 2: f16 ? pick_gu<2, true>(L, s) : pick_gu<2, false>(L, s); break;
        case 3: f16 ? pick_gu<3, true>(L, s) : pick_gu<3, false>(L, s); break;
        default: f16 ? pick_gu<4, true>(L, s) : pick_gu<4, false>(L, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_down_few(const ExpertLaunch& L, hipStream_t s) {
    if (L.table != nullptr || !few_ok(L.hidden, L.inter, L.n_tokens, L.max_lds)) return hipErrorInvalidValue;
    const bool full = L.inter / kKB == 16;
    switch (few_tiles(L.n_tokens)) {
        case 1: full ? go_dn<4, 1>(L, s) : go_dn<1, 1>(L, s); break;
        case 2: full ? go_dn<4, 2>(L, s) : go_dn<1, 2>(L, s); break;
        case 3: full ? go_dn<4, 3>(L, s) : go_dn<1, 3>(L, s); break;
        default: full ? go_dn<4, 4>(L, s) : go_dn<1, 4>(L, s); break;
    }
    return hipGetLastError();
}

}  // namespace cx
