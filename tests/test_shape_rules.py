"""The rules of csrc/cx_shapes.h over ranges of sizes, on the host: the scratch a
call asks for covers what its kernels use and every call with fewer tokens."""
from __future__ import annotations

import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "constellation_amd" / "csrc"

SOURCE = r"""
#include "cx_shapes.h"
using namespace cx;
extern "C" {
void expert(int t, int h, int i, int lds, size_t* out) {
    const ExpertScratch z = expert_scratch(t, h, i, lds);
    out[0] = z.bytes; out[1] = z.lo_bytes;
}
size_t call(int t, int h, int i, int lds, int dma) {
    return expert_call_bytes(expert_route(t, h, i, lds, dma, dma, dma).path, t, i);
}
int small(int h, int i) { return expert_small_shape(h, i); }
size_t few_bytes(int t, int i) { return few_scratch_bytes(t, i); }
int few(int h, int i, int t, int lds) { return few_ok(h, i, t, lds); }
int aligned(size_t p) { return dma_aligned((const void*)p); }
void route(int t, int h, int i, int lds, int x, int gu, int dn, int* out) {
    const ExpertRoute r = expert_route(t, h, i, lds, x, gu, dn);
    out[0] = r.path; out[1] = r.pp_gate_up; out[2] = r.pp_down; out[3] = r.np_lds;
}
int big(int h, int i, int n, int sh) { return big_min_pairs(h, i, n, sh, 256); }
int few_lds(int t) { return few_gu_lds(few_tiles(t)); }
int slices(int t, int h, int e) { return route_slices(t, h, e); }
void router(int t, int h, int e, int decode, int inter, size_t* out) {
    const RouteScratch z = route_scratch(t, h, e, decode, inter);
    out[0] = z.part; out[1] = z.scores; out[2] = z.gu_part; out[3] = z.bytes;
}
size_t buffer(int t, int k, int e, int sh) { return plan_buffer_bytes(t, k, e, sh); }
size_t plan(int t, int k, int e, int sh, int cap, int dense) {
    PlanSizes z = plan_sizes(t, k, e, sh);
    z.max_items = dense ? z.max_slots : z.max_slots + (z.max_pairs + cap - 1) / cap;
    return plan_bytes(z, t, k, dense);
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cc").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(d / "rules.cc"), "-o", str(d / "rules.so")], check=True)
    L = C.CDLL(str(d / "rules.so"))
    for f in ("few_bytes", "call", "buffer", "plan"):
        getattr(L, f).restype = C.c_size_t
    return L


@pytest.mark.parametrize("lds", [160 << 10, 64 << 10])
@pytest.mark.parametrize("H,I", [(7168, 2048), (1024, 512), (512, 512), (7168, 512), (4096, 1536), (2048, 768)])
def test_expert_scratch_never_shrinks(rules, H, I, lds):
    last = (0, 0)
    for T in range(1, 700):
        out = (C.c_size_t * 2)()
        rules.expert(T, H, I, lds, out)
        assert out[0] >= last[0] and out[1] >= last[1], (T, last, list(out))
        last = tuple(out)
        for dma in (0, 1):
            need = rules.call(T, H, I, lds, dma)
            if T <= 4 and rules.small(H, I):
                assert need == 16 * T * I  # two k-parts of gate and up, fp32
            elif dma and rules.few(H, I, T, lds):
                assert need == rules.few_bytes(T, I)
            else:
                assert need == (2 * T * I + 255) // 256 * 256 + 2 * T * I
                if T > 64:  # a buffer for each plane
                    assert out[1] == 2 * T * I
                    need = 2 * T * I
            assert need <= out[0], (T, need, list(out))


@pytest.mark.parametrize("lds", [160 << 10, 96 << 10, 64 << 10, 16 << 10])
def test_few_token_kernels_fit_the_lds(rules, lds):
    """5..64 tokens where a workgroup can have the LDS, else the other kernels."""
    for T in range(1, 80):
        assert bool(rules.few(7168, 2048, T, lds)) == (5 <= T <= 64 and rules.few_lds(T) <= lds), T


@pytest.mark.parametrize("H,I", [(7168, 2048), (1024, 512), (4096, 1536), (640, 384)])
def test_wide_loads_only_from_aligned_rows(rules, H, I):
    """Rows of x or weights that do not start on 16 bytes take the kernels with
    plain loads (and the others' are not changed by them)."""
    assert [rules.aligned(p) for p in (0, 16, 2, 4, 8, 0x7f0000000010, 0x7f000000000e)] == [1, 1, 0, 0, 0, 1, 0]
    small, tiles, few = 1, 2, 3

    def route(T, *dma):
        out = (C.c_int * 4)()
        rules.route(T, H, I, 160 << 10, *dma, out)
        return tuple(out)

    for T in list(range(1, 140)) + [1000]:
        best = route(T, 1, 1, 1)
        pp = H % 256 == 0 and T > 16 and best[0] == tiles
        assert best[0] == (few if rules.few(H, I, T, 160 << 10) else small if T <= 4 and rules.small(H, I) else tiles)
        assert best[1:3] == (pp, pp)
        assert best[3] == (T if T <= (3 if H == 7168 else 4) and H % 512 == 0 else 0)
        got = route(T, 0, 1, 1)
        assert got == (small if best[0] == small else tiles, 0, H % 256 == 0 and T > 16, 0), T
        if not best[0] == few:
            assert route(T, 1, 0, 1) == best[:1] + (0,) + best[2:]
            assert route(T, 1, 1, 0) == best[:2] + (0,) + best[3:]


@pytest.mark.parametrize("H,E", [(7168, 256), (1024, 64), (640, 72), (384, 40), (1000, 8)])
@pytest.mark.parametrize("decode,inter", [(0, 0), (1, 0), (1, 512)])
def test_router_scratch_never_shrinks(rules, H, E, decode, inter):
    last = 0
    for T in range(1, 600):
        out = (C.c_size_t * 4)()
        rules.router(T, H, E, decode, inter, out)
        part, scores, gu, end = out
        assert end >= last, T
        last = end
        assert not any(p % 256 for p in (part, scores, gu)) and part >= 8 * T * E
        if T > 16 or not decode:
            assert scores - part >= 8 * rules.slices(T, H, E) * T * E, T
        if decode:
            assert gu - scores >= 16 * E and end - gu >= 16 * min(T, 8) * inter, T


@pytest.mark.parametrize("H,I,n,shared,pairs", [
    (7168, 2048, 256, 1, 20), (7168, 2048, 127, 1, 20), (7168, 2048, 64, 0, 20), (7168, 2048, 4, 0, 20),
    (7168, 2048, 64, 1, 64), (7168, 2048, 16, 1, 64), (7168, 2048, 15, 1, 20),  # the shared expert's items last
    (7168, 512, 256, 1, 64), (7168, 512, 255, 1, 80), (1024, 2048, 64, 0, 80), (1024, 512, 32, 1, 80), (512, 512, 31, 0, 128),  # few blocks
    (2048, 768, 128, 1, 20), (4096, 1536, 8, 1, 20), (2048, 512, 64, 1, 20)])  # no 64-pair kernels
def test_pairs_per_expert_of_128_pair_items(rules, H, I, n, shared, pairs):
    """The least pairs per resident expert for 128-pair items, on 256 CUs."""
    assert rules.big(H, I, n, shared) == pairs


@pytest.mark.parametrize("H,E,least,most", [(7168, 256, 4, 256), (7168, 384, 4, 160), (1024, 512, 5, 128),
                                            (2048, 64, 4, 256), (640, 384, 4, 256), (1000, 8, 4, 0)])
def test_router_tiles_in_one_round(rules, H, E, least, most):
    """The 16 x 16 tiles of the router's logits up to one round of 256 CUs, or 256
    tokens where the 16 x 32 tiles do not take the width."""
    for T in range(1, 300):
        assert bool(rules.slices(T, H, E)) == (least <= T <= most), T


@pytest.mark.parametrize("E,K", [(256, 8), (64, 8), (4, 2), (128, 1), (512, 64)])
@pytest.mark.parametrize("shared", [0, 1])
def test_plan_buffer_never_shrinks(rules, E, K, shared):
    last = 0
    for T in range(1, 1500):
        got = rules.buffer(T, K, E, shared)
        assert got >= last, T
        last = got
        forms = [(64, 0), (128, 0)] if T > 16 else [(16, 0), (16, 1), (128, 0)]
        assert all(rules.plan(T, K, E, shared, cap, dense) <= got for cap, dense in forms), T
