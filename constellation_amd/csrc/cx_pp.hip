// cx_pp.hip — kernels and launchers of the ping-pong grouped GEMM (cx_pp.h).
#include "cx_pp.h"

namespace cx {
namespace {

template <bool F16>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_gu_pp(ExpertLaunch L) {
    extern __shared__ __attribute__((aligned(16))) unsigned char pp_lds[];
    pp_gate_up<F16>(L, pp_lds);
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_dn_pp(ExpertLaunch L) {
    extern __shared__ __attribute__((aligned(16))) unsigned char pp_lds[];
    pp_down(L, pp_lds);
}

// Every (item, row tile) of the plan's bound, rounded up to whole XCD rows
// (pp_tile maps the tiles that exist).
dim3 pp_grid(const ExpertLaunch& L, int row_tiles) { return dim3((L.max_items * row_tiles + 7) / 8 * 8); }

}  // namespace

bool pp_ok(int hidden, int inter, int max_lds) {
    return inter % kPpRowsGu == 0 && hidden % kPpRowsDn == 0 && hidden / kKB >= kPpMinBlocks &&
           inter / kKB >= kPpMinBlocks && max_lds >= kPpLds;
}

hipError_t launch_gate_up_pp(const ExpertLaunch& L, hipStream_t s) {
    if (L.table == nullptr || !pp_ok(L.hidden, L.inter, L.max_lds)) return hipErrorInvalidValue;
    const dim3 grid = pp_grid(L, L.inter / kPpRowsGu), block(512);
    if (L.in_dtype == CX_DTYPE_FP16) cx_launch(k_gu_pp<true>, grid, block, kPpLds, s, L);
    else cx_launch(k_gu_pp<false>, grid, block, kPpLds, s, L);
    return hipGetLastError();
}

hipError_t launch_down_pp(const ExpertLaunch& L, hipStream_t s) {
    if (L.table == nullptr || !pp_ok(L.hidden, L.inter, L.max_lds)) return hipErrorInvalidValue;
    cx_launch(k_dn_pp, pp_grid(L, L.hidden / kPpRowsDn), dim3(512), kPpLds, s, L);
    return hipGetLastError();
}

}  // namespace cx
