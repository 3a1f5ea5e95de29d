"""Which kernels the 16-bit launches are made of, asked of the library on the host: the cases of the GPU tests that are about one
kernel reach it, and plans hold where they were measured."""
import ctypes

import pytest
import torch

from simplical_attn_amd import _lib
from tests import test_gpu_bwd_kp_lone, test_gpu_bwd_kv, test_gpu_fwd_lone, test_gpu_split_fwd_lone, test_gpu_split_kp_lone, test_gpu_split_kv_lone


def _ask(name, B, N, H, D, w1, w2, force=None):
    f = getattr(_lib.load(), name)          # (functions of namespace sa2, declared in csrc/sa2_common.h)
    args = [ctypes.c_int(x) for x in (B, N, H, D, min(w1, N - 1), min(w2, N - 1))]
    return f(*args) if force is None else f(*args, ctypes.c_bool(force))


def forward_route(B, N, H, D, w1, w2, force=False):
    """(pre-pass, two units per wavefront, shares)"""
    r = _ask("_ZN3sa214mfma_fwd_routeEiiiiiib", B, N, H, D, w1, w2, force)
    return bool(r & 1), bool(r & 2), r >> 8


def kp_route(B, N, H, D, w1, w2, force=False):
    """(pre-pass, one wavefront per SIMD, segments)"""
    r = _ask("_ZN3sa213mfma_kp_routeEiiiiiib", B, N, H, D, w1, w2, force)
    return bool(r & 1), bool(r & 2), r >> 8


def kv_route(B, N, H, D, w1, w2):
    """(32-row K blocks per wavefront, shares)"""
    r = _ask("_ZN3sa213mfma_kv_routeEiiiiii", B, N, H, D, w1, w2)
    return r & 255, r >> 8


def split_route(what, dtype, B, N, H, D, w1, w2):
    """Plane-split kernels: (one wavefront per SIMD, shares or segments)"""
    f = getattr(_lib.load(), "_ZN3sa2%dsplit_%s_routeEiiiiiii" % (len("split__route" + what), what))
    code = {torch.float32: _lib.SA2_F32, torch.bfloat16: _lib.SA2_BF16, torch.float16: _lib.SA2_F16}[dtype]
    r = f(*[ctypes.c_int(x) for x in (B, N, H, D, min(w1, N - 1), min(w2, N - 1), code)])
    return bool(r & 1), r >> 8


def _cases(test):
    return next(m for m in test.pytestmark if m.name == "parametrize").args[1]


def _types(test):
    return next(m for m in test.pytestmark if m.name == "parametrize" and m.args[0] == "dtype,D").args[1]


@pytest.mark.parametrize("B,N,H,D,w1,w2,lone", [
    (1, 4096, 8, 64, 512, 0, False),        # one delta: half of what a wavefront with two units computes is thrown away
    (1, 4096, 16, 64, 512, 2, False), (1, 4096, 16, 64, 512, 6, True), (2, 2048, 8, 64, 512, 32, True),
    (1, 2600, 4, 64, 150, 40, False), (1, 6950, 1, 64, 226, 40, False), (1, 969, 7, 64, 272, 20, True),
    (1, 4096, 16, 128, 512, 1, False), (1, 3000, 8, 128, 500, 31, False), (1, 8192, 16, 128, 512, 32, True), (1, 32768, 8, 128, 1024, 64, True),
])
def test_kp_side_by_keys_deltas_and_grid(B, N, H, D, w1, w2, lone):
    assert kp_route(B, N, H, D, w1, w2)[1] == lone


def test_kp_cases_reach_the_kernel():
    cases = _cases(test_gpu_bwd_kp_lone.test_kp_side_matches_the_fma_kernels)
    at = next(i for i, c in enumerate(cases) if c[1:4] == (1, 2051, 20))
    routes = {c[1:7]: kp_route(*c[1:7]) for c in cases[at:]}
    assert all(lone for _, lone, _ in routes.values())
    assert routes[1, 1003, 26, 128, 900, 40][0] and routes[1, 900, 8, 128, 899, 200][2] > 1
    for D, N, heads, w1, w2 in _cases(test_gpu_bwd_kp_lone.test_layouts_and_half_open_windows):
        assert kp_route(1, N, heads, D, w1 - 1, w2 - 1)[1]


def test_kp_side_of_narrower_windows():
    """by the keys per unit that a round has room for, and at head_dim 128 by the grid"""
    cases = _cases(test_gpu_bwd_kp_lone.test_narrower_windows_of_many_deltas)
    routes = {c[1:7]: kp_route(*c[1:7]) for c in cases}
    assert all(lone for _, lone, _ in routes.values()) and routes[1, 353, 8, 64, 2000, 130][2] > 1
    for not_taken in ((1, 3000, 8, 64, 150, 9), (1, 4096, 16, 64, 256, 3), (1, 2048, 4, 64, 128, 32), (1, 1200, 6, 128, 260, 31),
                      (1, 8192, 16, 128, 256, 4), (1, 8192, 16, 128, 192, 31)):
        assert not kp_route(*not_taken)[1]


def test_k2_row_cases_reach_the_kernel():
    routes = {c[4:6] + c[6:7]: kp_route(*c[1:7]) for c in _cases(test_gpu_bwd_kp_lone.test_k2_rows_in_both_forms)}
    assert all(lone for _, lone, _ in routes.values()) and routes[128, 900, 24][0] and routes[64, 500, 32][0]
    assert all(segments == 1 for _, _, segments in routes.values())


def test_forward_cases_reach_the_kernel():
    t = test_gpu_fwd_lone
    routes = [(c[0], c[4], *forward_route(*c[1:7])) for c in _cases(t.test_forward_matches_the_fma_kernels)]
    reached = {(dtype, D, left) for dtype, D, left, two, shares in routes if two}
    assert {(t.BF, 64, False), (t.FP, 64, False), (t.BF, 64, True), (t.BF, 128, False), (t.FP, 128, False), (t.BF, 128, True)} <= reached
    assert any(two and shares > 1 for _, _, _, two, shares in routes)
    far = [m.args[1] for f in (t.test_logits_that_leave_the_reference_point_behind, t.test_logits_that_leave_the_reference_point_behind_in_long_sweeps_and_shares)
           for m in f.pytestmark if "," in m.args[0]]
    routes = {(D, w2, heads): forward_route(1, 470, heads, D, 300, w2) for D, w2, heads in far[0] + far[1]}
    assert routes[64, 5, 20][1:] == (True, 1) and routes[64, 16, 60][:2] == (True, True) and routes[128, 30, 300][:2] == (False, True)
    assert routes[128, 24, 400][:2] == (True, True) and routes[64, 130, 6][1] and routes[64, 130, 6][2] > 1
    for c in _cases(t.test_second_pass_on_widely_spread_logits):
        assert forward_route(*c[:6])[1]
    for D, heads, w2 in _cases(t.test_a_key_that_is_not_a_number_stays_in_its_window):
        assert forward_route(1, 600, heads, D, 230, w2)[1]
    assert forward_route(1, 1500, 6, 64, 199, 19)[1] and forward_route(1, 4100, 32, 128, 299, 23)[1]      # (test_layouts_and_half_open_windows)


def test_kv_cases_have_both_geometries_and_shares():
    routes = {c[1:7]: kv_route(*c[1:7]) for c in _cases(test_gpu_bwd_kv.test_k_side_matches_the_fma_kernels)}
    assert routes[4, 520, 64, 64, 300, 3] == (2, 1) and routes[1, 400, 130, 64, 390, 0] == (2, 1) and routes[1, 129, 1, 64, 40, 33][1] > 1
    assert routes[2, 17, 4, 64, 16, 16] == (1, 8) and routes[1, 31, 2, 32, 20, 30][1] > 1


@pytest.mark.parametrize("B,N,H,D,w1,w2,want", [
    (2, 17, 4, 64, 128, 24, (1, 8)), (2, 17, 4, 16, 128, 24, (1, 8)), (2, 9, 4, 64, 128, 24, (1, 1)),       # one query block
    (5, 448, 29, 32, 816, 96, (1, 2)), (2, 2048, 8, 64, 512, 32, (2, 2)), (1, 8192, 16, 128, 512, 32, (1, 1)),
])
def test_k_side_plan(B, N, H, D, w1, w2, want):
    assert kv_route(B, N, H, D, w1, w2) == want


def test_plane_split_forward_cases_reach_both_kernels():
    """Two units per wavefront where their test is about them: rounds of one to eight units, short sweeps, shares, moved reference points."""
    t = test_gpu_split_fwd_lone
    for dtype, D in t.TYPES:
        route = lambda B, N, H, w1, w2: split_route("fwd", dtype, B, N, H, D, w1, w2)
        matches = {c[:5]: route(*c[:5]) for c in _cases(t.test_forward_matches_the_fma_kernels)}
        many = [route(*c[:5]) for c in _cases(t.test_short_sequences_of_many_heads)]
        if D <= 32:
            assert not any(lone for lone, _ in list(matches.values()) + many)
            continue
        assert all(lone for lone, _ in many)
        two = (dtype, D) != (t.FP, 80)                      # (there shares of up to twenty deltas have one unit per wavefront)
        for case in ((1, 520, 2, 95, 33), (1, 640, 30, 70, 40), *(((1, 200, 1, 500, 8), (1, 161, 1, 3, 12)) if D <= 64 else ())):
            assert matches[case][0]
        assert matches[1, 520, 2, 95, 33][1] > 1 and not matches[1, 33, 1, 0, 0][0]
        assert route(1, 470, 2, 300, 12)[0] == two and route(1, 470, 40, 300, 20)[0] and route(1, 400, 6, 150, 20)[0]
        assert route(2, 150, 8, 149, 9)[0] == two and route(2, 150, 8, 149, 40)[0] and route(2, 150, 1, 149, 30)[0] and route(2, 64, 70, 63, 8)[0]


@pytest.mark.parametrize("dtype,D,shape,lone", [
    (torch.float32, 64, (1, 826, 1, 31, 2), False), (torch.float32, 64, (1, 131, 46, 90, 4), False), (torch.float32, 64, (1, 388, 7, 405, 4), True),
    (torch.float32, 64, (1, 1052, 19, 49, 5), True), (torch.float32, 64, (1, 67, 8, 52, 9), False), (torch.float32, 64, (1, 67, 53, 23, 23), True),
    (torch.float32, 64, (2, 2048, 8, 512, 32), True), (torch.float16, 48, (1, 378, 31, 64, 6), False), (torch.float16, 48, (1, 388, 7, 387, 5), True),
    (torch.float16, 48, (1, 4221, 4, 766, 2), True), (torch.float16, 80, (1, 709, 11, 12, 3), False), (torch.float16, 80, (1, 5041, 4, 256, 3), True),
    (torch.bfloat16, 40, (1, 274, 1, 27, 5), False), (torch.bfloat16, 40, (1, 1052, 19, 49, 5), True), (torch.bfloat16, 96, (1, 45, 16, 16, 1), False),
    (torch.bfloat16, 96, (1, 826, 1, 31, 2), True), (torch.bfloat16, 96, (1, 2048, 8, 255, 31), True)])
def test_plane_split_forward_by_deltas_and_sweep(dtype, D, shape, lone):
    B, N, H, w1, w2 = shape
    assert split_route("fwd", dtype, B, N, H, D, w1, w2)[0] == lone


def test_plane_split_kp_cases_reach_both_kernels():
    t = test_gpu_split_kp_lone
    for dtype, D in _types(t.test_kp_side_matches_the_fma_kernels):
        route = lambda c: split_route("kp", dtype, c[0], c[1], c[2], D, c[3], c[4])
        assert all(route(c)[0] for c in _cases(t.test_short_sequences_of_many_heads))
        matches = {c[:5]: route(c) for c in _cases(t.test_kp_side_matches_the_fma_kernels)}
        assert matches[1, 640, 16, 70, 400][0] and matches[1, 640, 16, 70, 400][1] > 1 and matches[1, 700, 40, 129, 3][0]
        assert matches[1, 33, 1, 0, 0][0] == ((dtype, D) in ((t.F32, 64), (t.BF, 72), (t.BF, 96)))


@pytest.mark.parametrize("dtype,D,shape,lone", [
    (torch.float32, 16, (1, 1314, 1, 17, 10), False), (torch.float32, 16, (1, 599, 1, 465, 1), True), (torch.float32, 32, (1, 119, 2, 23, 1), False),
    (torch.float32, 64, (1, 119, 2, 23, 1), True), (torch.float16, 48, (1, 225, 2, 89, 10), False), (torch.float16, 80, (1, 773, 1, 236, 1), False),
    (torch.float16, 80, (1, 2048, 8, 255, 31), True), (torch.bfloat16, 40, (1, 58, 1, 35, 12), False), (torch.bfloat16, 40, (1, 381, 2, 380, 9), True),
    (torch.bfloat16, 96, (1, 58, 1, 35, 12), True)])
def test_plane_split_kp_side_by_grid_and_sweep(dtype, D, shape, lone):
    B, N, H, w1, w2 = shape
    assert split_route("kp", dtype, B, N, H, D, w1, w2)[0] == lone


def test_plane_split_kv_cases_reach_both_kernels():
    t = test_gpu_split_kv_lone
    for dtype, D in _types(t.test_k_side_matches_the_fma_kernels):
        routes = {c[:5]: split_route("kv", dtype, c[0], c[1], c[2], D, c[3], c[4]) for c in _cases(t.test_k_side_matches_the_fma_kernels)}
        assert all(lone == (dtype != t.FP or N > 80 or w2 >= 20) for (B, N, H, w1, w2), (lone, _) in routes.items())
        assert routes[1, 520, 2, 95, 33][1] > 1 and routes[3, 40, 5, 40, 39][0]
