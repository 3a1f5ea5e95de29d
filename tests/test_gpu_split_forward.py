"""Forward launches whose rounds are shared by several workgroups (short sequences with wide K' windows): the partial
outputs, their merge and the second pass of an overflowed block, against the CPU oracle; sa2_forward without a workspace
computes the same problem in one workgroup per query block."""
import pytest
import torch

from oracle import simplicial_oracle as orc
from simplical_attn_amd import _lib
from tests.util import assert_close_rel, make_inputs, oracle_all

pytestmark = pytest.mark.gpu
CODE = {torch.float32: _lib.SA2_F32, torch.bfloat16: _lib.SA2_BF16, torch.float16: _lib.SA2_F16}
BAR = {torch.bfloat16: 2e-2, torch.float16: 1e-2, torch.float32: 1e-5}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [(1, 130, 2, 64, 40, 60, True), (2, 97, 1, 128, 200, 47, False), (1, 256, 1, 32, 33, 255, True),
                                  (1, 77, 3, 16, 20, 33, True), (1, 33, 1, 96, 8, 40, True)])
@pytest.mark.parametrize("scale", [None, 6.0])
def test_shares_of_the_rounds_merge_to_the_oracle(dtype, case, scale):
    """scale 6: logits of hundreds, so that blocks overflow their first reference point and take the second pass."""
    import simplical_attn_amd as sa
    lib = _lib.load()
    B, N, H, D, w1, w2, inclusive = case
    assert lib.sa2_fwd_workspace_bytes(B, N, H, D, w1, w2, CODE[dtype], int(inclusive), 0) > 0
    host = make_inputs(B, N, H, D, seed=N, dtype=dtype)
    x = [t.cuda() for t in host[:5]]
    out, lse = sa.simplicial_forward(*x, w1, w2, scale, 0.1, -0.2, window_inclusive=inclusive)
    want = oracle_all(host, w1, w2, scale, 0.1, -0.2, inclusive=inclusive)
    # (16-bit logits of hundreds carry absolute errors of their rounding: the largest weight may change hands)
    if scale is None or dtype == torch.float32:
        assert_close_rel(out, want["out"], BAR[dtype] if scale is None else 2e-4, "out")
    assert torch.isfinite(out.float()).all()
    assert_close_rel(lse, want["lse"], BAR[dtype] if scale is None or dtype != torch.float32 else 1e-5, "lse")
    o1, l1 = torch.empty_like(out), torch.empty_like(lse)
    strides = _lib.stride_array([(t.stride(0), t.stride(1), t.stride(2)) for t in (*x, o1)])
    _lib.check(lib.sa2_forward(*[t.data_ptr() for t in x], o1.data_ptr(), l1.data_ptr(), B, N, H, D, strides, w1, w2,
                               D ** -0.5 if scale is None else scale, 0.1, -0.2, CODE[dtype], int(inclusive), 0,
                               torch.cuda.current_stream().cuda_stream))
    assert_close_rel(out, o1.float().cpu(), {torch.float32: 1e-5 if scale is None else 2e-4}.get(dtype, 1e-2), "out, shared against whole")
    assert_close_rel(lse, l1.cpu(), 1e-5 if dtype == torch.float32 else 1e-3, "lse, shared against whole")
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 32), (torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 96),
                                     (torch.bfloat16, 256), (torch.float32, 64), (torch.float32, 96)])
def test_a_query_that_is_not_a_number_stays_one_through_the_merge(dtype, D):
    import simplical_attn_amd as sa
    assert _lib.load().sa2_fwd_workspace_bytes(1, 160, 1, D, 40, 60, CODE[dtype], 1, 0) > 0
    x = [t.cuda() for t in make_inputs(1, 160, 1, D, seed=2, dtype=dtype, with_dout=False)]
    x[0][:, 70] = float("nan")
    out, _ = sa.simplicial_forward(*x, 40, 60)
    rows = out[0, :, 0].isnan()
    assert rows[70].all() and rows.sum().item() == D


@pytest.mark.parametrize("dtype,case,shares", [
    (torch.float32, (1, 100, 1, 16, 70, 8, True), 2),        # the second share has one unit
    (torch.float32, (1, 128, 2, 64, 32, 16, True), 3),
    (torch.float32, (2, 67, 3, 128, 30, 9, True), 3),
    (torch.float32, (1, 1021, 4, 32, 70, 23, True), 2),     # three rounds in two shares: as many as there are CUs for
    (torch.bfloat16, (1, 63, 2, 96, 40, 9, False), 3),    # rounds of four units
    (torch.bfloat16, (1, 97, 2, 96, 40, 12, False), 2),
    (torch.float16, (1, 300, 5, 80, 20, 22, True), 3),
    (torch.float16, (2, 130, 2, 80, 40, 11, True), 3),      # ... and here
    (torch.bfloat16, (1, 200, 2, 64, 150, 20, True), 3),
    (torch.float16, (1, 128, 2, 128, 100, 12, True), 2),
    (torch.bfloat16, (1, 70, 2, 256, 16, 11, True), 3),
])
def test_small_grids_share_two_or_three_rounds(dtype, case, shares):
    """As above; a workspace that is too small for the shares leaves the launch whole."""
    import simplical_attn_amd as sa
    lib = _lib.load()
    B, N, H, D, w1, w2, inclusive = case
    width = next(w for w in (32, 64, 96, 128, 256) if w >= D)
    assert lib.sa2_fwd_workspace_bytes(B, N, H, D, w1, w2, CODE[dtype], int(inclusive), 0) == shares * B * H * N * (width + 2) * 4
    test_shares_of_the_rounds_merge_to_the_oracle(dtype, case, None)
    x = [t.cuda() for t in make_inputs(B, N, H, D, seed=N, dtype=dtype)[:5]]
    small = torch.empty(256, dtype=torch.uint8, device="cuda")
    got = []
    for workspace in (None, small):
        o, l = torch.empty_like(x[0]), torch.empty(B, H, N, device="cuda")
        strides = _lib.stride_array([(t.stride(0), t.stride(1), t.stride(2)) for t in (*x, o)])
        _lib.check(lib.sa2_forward_ws(*[t.data_ptr() for t in x], o.data_ptr(), l.data_ptr(), workspace.data_ptr() if workspace is not None else None,
                                      256 if workspace is not None else 0, B, N, H, D, strides, w1, w2, D ** -0.5, 0.1, -0.2, CODE[dtype],
                                      int(inclusive), 0, torch.cuda.current_stream().cuda_stream))
        got.append((o, l))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 96), (torch.float16, 48), (torch.float32, 128)])
@pytest.mark.parametrize("w2", [0, 40])
def test_lse_of_small_logits(dtype, D, w2):
    """Queries with one key each (the first ones: one K' row too) and logits of 1e-3: LSE is the logit plus the logarithm of the K' rows,
    to the roundings of both (2^-24 of each; the 1e-8 of the sum is lost beside 1)."""
    import simplical_attn_amd as sa
    host = make_inputs(1, 200, 4, D, seed=D, dtype=dtype)
    x = [t.cuda() for t in host[:5]]
    lse = sa.simplicial_forward(*x, 0, w2, 1e-4)[1]
    want = orc.forward_windowed(*[t.double() for t in host[:5]], 0, w2, 1e-4)[1]
    assert ((lse.double().cpu() - want).abs() <= 1.2e-8 + 2.5e-7 * want.abs()).all()
