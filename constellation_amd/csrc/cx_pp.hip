// cx_pp.hip — kernels and launchers of the ping-pong grouped GEMM (cx_pp.h).
#include "cx_pp.h"

namespace cx {
namespace {

template <bool F16, bool SINGLE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_gu_pp(ExpertLaunch L) {
    extern __shared__ __attribute__((aligned(16))) unsigned char pp_lds[];
    pp_gate_up<F16, SINGLE>(L, pp_lds);
}

template <bool SINGLE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_dn_pp(ExpertLaunch L) {
    extern __shared__ __attribute__((aligned(16))) unsigned char pp_lds[];
    pp_down<SINGLE>(L, pp_lds);
}

// Tokens per item for one expert over n_tokens: the workgroups run in rounds of
// n_cu, each as long as an item of that many column tiles takes; the count with
// the least rounds x time, the larger of equals (fewer reads of the weights).
// us[n - 1]: an item of n column tiles alone on its CU at hidden 7168, inter
// 2048, from 17 to 4096 tokens of one expert at every count; only their ratios
// matter (rows of other lengths take the same counts; at ten shapes from 512 x 512
// to 4096 x 1536 no call of 17 to 4096 tokens was slower than with the 64-token items
// before).  At 300 tokens gate/up takes 35 us with 2 tiles and 43 with 4, down 23
// with 3 and 35 with 2; at 1500 80 with 6 and 96 with 4.
constexpr int kPpUsGu[kPpMaxTiles] = {27, 33, 40, 43, 56, 65, 74, 84};
constexpr int kPpUsDn[kPpMaxTiles] = {13, 17, 22, 24, 38, 38, 45, 45};

int pp_single_cap(int n_tokens, int row_tiles, int n_cu, const int (&us)[kPpMaxTiles]) {
    int best = 1;
    int64_t least = INT64_MAX;
    for (int n = 1; n <= kPpMaxTiles; ++n) {
        const int64_t items = (n_tokens + n * kTileTok - 1) / (n * kTileTok);
        const int64_t t = (items * row_tiles + n_cu - 1) / n_cu * us[n - 1];
        if (t <= least) {
            least = t;
            best = n;
        }
    }
    return best * kTileTok;
}

// Every (item, row tile) of the launch, rounded up to whole XCD rows (pp_tile
// maps the tiles that exist).
dim3 pp_grid(const ExpertLaunch& L, int row_tiles) {
    const int items = L.table != nullptr ? L.max_items : (L.n_tokens + L.item_cap - 1) / L.item_cap;
    return dim3((items * row_tiles + 7) / 8 * 8);
}

}  // namespace

hipError_t launch_gate_up_pp(const ExpertLaunch& L0, hipStream_t s) {
    ExpertLaunch L = L0;
    if (!pp_ok(L.hidden, L.inter, L.max_lds)) return hipErrorInvalidValue;
    const int row_tiles = L.inter / kPpRowsGu;
    const bool f16 = L.in_dtype == CX_DTYPE_FP16;
    const dim3 block(512);
    if (L.table != nullptr) {
        const dim3 grid = pp_grid(L, row_tiles);
        if (f16) cx_launch((k_gu_pp<true, false>), grid, block, kPpLds, s, L);
        else cx_launch((k_gu_pp<false, false>), grid, block, kPpLds, s, L);
    } else {
        L.item_cap = pp_single_cap(L.n_tokens, row_tiles, L.n_cu > 0 ? L.n_cu : 256, kPpUsGu);
        const dim3 grid = pp_grid(L, row_tiles);
        if (f16) cx_launch((k_gu_pp<true, true>), grid, block, kPpLds, s, L);
        else cx_launch((k_gu_pp<false, true>), grid, block, kPpLds, s, L);
    }
    return hipGetLastError();
}

hipError_t launch_down_pp(const ExpertLaunch& L0, hipStream_t s) {
    ExpertLaunch L = L0;
    if (!pp_ok(L.hidden, L.inter, L.max_lds)) return hipErrorInvalidValue;
    const int row_tiles = L.hidden / kPpRowsDn;
    const dim3 block(512);
    if (L.table != nullptr) {
        cx_launch((k_dn_pp<false>), pp_grid(L, row_tiles), block, kPpLds, s, L);
    } else {
        L.item_cap = pp_single_cap(L.n_tokens, row_tiles, L.n_cu > 0 ? L.n_cu : 256, kPpUsDn);
        cx_launch((k_dn_pp<true>), pp_grid(L, row_tiles), block, kPpLds, s, L);
    }
    return hipGetLastError();
}

}  // namespace cx
