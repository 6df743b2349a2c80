"""The grouped GEMM's tile and K-loop edges: 1 to 5 K steps (the loop's prologue,
its last two steps and both parities), groups that end inside each 64-row block
of a 256-row tile, column counts that are not whole tiles.

bf16: against the float64 product within one bf16 rounding plus the fp32
summation bound K * 2^-24 * sum |a||w|.  int8: the integer product dequantised in
the documented order, exactly.  fp8: the bf16 kernel on the dequantised rows,
exactly (the same sums in the same order)."""
import pytest
import torch

import moe_route as M

pytestmark = pytest.mark.gpu

BASE = [1, 64, 129, 129, 320, 577, 833, 1100]  # 1, 63, 65, 0, 191, 257, 256, 267 rows
# 137 rows a group on average; with empty groups added, few enough that short tiles
# (64 and 128 rows) take the ring loop
EMPTY = [0, 8]


def groups(ends, rows):
    lo = 0
    for g, hi in enumerate(ends):
        yield g, lo, hi
        lo = hi


def make(K, N, dev, seed, empty):
    ENDS = BASE + BASE[-1:] * empty
    g = torch.Generator(device=dev).manual_seed(seed)
    rows = ENDS[-1] + 30  # the last rows belong to no group
    a = torch.randn(rows, K, generator=g, device=dev).bfloat16()
    w = torch.randn(len(ENDS), N, K, generator=g, device=dev).bfloat16()
    return a, w, torch.tensor(ENDS, dtype=torch.int32, device=dev), ENDS


@pytest.mark.parametrize("empty", EMPTY)
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("N", [256, 264, 131])
def test_bf16(cuda, K, N, empty):
    a, w, offs, ENDS = make(K, N, cuda, K + N, empty)
    out = torch.full((a.shape[0], N), 7.0, dtype=torch.bfloat16, device=cuda)
    M.grouped_gemm(a, w, offs, out=out)
    for g, lo, hi in groups(ENDS, a.shape[0]):
        ref = a[lo:hi].double() @ w[g].double().t()
        mag = a[lo:hi].double().abs() @ w[g].double().abs().t()
        err = (out[lo:hi].double() - ref).abs()
        assert bool((err <= ref.abs() * 2.0 ** -8 + K * 2.0 ** -24 * mag).all()), (g, lo, hi)
    assert bool((out[ENDS[-1]:] == 7.0).all())


@pytest.mark.parametrize("empty", EMPTY)
@pytest.mark.parametrize("K", [128, 256, 384, 512])
@pytest.mark.parametrize("N", [256, 131])
def test_int8(cuda, K, N, empty):
    a, w, offs, ENDS = make(K, N, cuda, K * 3 + N, empty)
    q, s = M.quant_rows_i8(a)
    wq, ws = M.quant_rows_i8(w)
    out = torch.full((a.shape[0], N), 7.0, dtype=torch.bfloat16, device=cuda)
    M.grouped_gemm_i8(q, s, wq, ws, offs, out=out)
    for g, lo, hi in groups(ENDS, a.shape[0]):
        acc = q[lo:hi].double() @ wq[g].double().t()  # exact integers
        ref = (acc.float() * (s[lo:hi, None] * ws[g][None])).bfloat16()
        assert torch.equal(out[lo:hi], ref), (g, lo, hi)
    assert bool((out[ENDS[-1]:] == 7.0).all())


@pytest.mark.parametrize("empty", EMPTY)
@pytest.mark.parametrize("K", [128, 256, 384])
@pytest.mark.parametrize("N", [256, 131])
@pytest.mark.parametrize("swiglu", [False, True])
def test_fp8_matches_bf16_on_dequantised_rows(cuda, K, N, swiglu, empty):
    a, w, offs, ENDS = make(K, N, cuda, K * 5 + N, empty)
    p = M.permute(a, torch.zeros(a.shape[0], 1, dtype=torch.int32, device=cuda), 1, fp8=True)
    q, s = p["xg"], p["scales"]
    deq = (q.view(torch.float8_e4m3fn).float().view(a.shape[0], -1, 128) * s[..., None]).view(
        a.shape[0], K).bfloat16()
    if swiglu:
        up = w.flip(0).contiguous()
        got, ref = M.grouped_swiglu_fp8(q, s, w, up, offs), M.grouped_swiglu(deq, w, up, offs)
    else:
        got, ref = M.grouped_gemm_fp8(q, s, w, offs), M.grouped_gemm(deq, w, offs)
    assert torch.equal(got[:ENDS[-1]], ref[:ENDS[-1]])
