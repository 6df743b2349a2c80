"""The grouped GEMM's ring kernel where a block takes two column tiles in a row (several
hundred tiles of few K steps): odd tile counts, a partial last tile, output rows that are
not whole 16-byte chunks, 1 to 16 K steps, groups of every kind of row tile in one call
(1 to 128 rows, 129 to 256, several tiles, none), more than 64 and more than 256 groups.

bf16: against the float64 product within one bf16 rounding plus the fp32 summation bound
K * 2^-24 * sum |a||w|; SwiGLU exactly as silu(gate) * up of a 256-row tile's sums, which
the same rows reach as one group.  int8: the integer product dequantised in the
documented order, exactly."""
import pytest
import torch

import moe_route as M

pytestmark = pytest.mark.gpu

# (groups, K, N): 4 .. 9 column tiles of 256; 256-byte, 1 KB and 2 KB weight rows
SHAPES = [(130, 64, 1024), (130, 128, 1288), (70, 512, 2304), (100, 1024, 1030), (300, 128, 1024)]
SIZES = [1, 16, 17, 33, 64, 65, 100, 128, 0, 5]


def ends_of(G, long_groups):
    """Group ends: sizes of one row tile, and with long_groups some of 129 rows and more."""
    rows = [SIZES[g % len(SIZES)] for g in range(G)]
    if long_groups:
        for g, r in ((3, 129), (G // 2, 256), (G // 2 + 1, 300), (G - 1, 700)):
            rows[g] = r
    return torch.tensor(rows).cumsum(0).tolist()


def inputs(G, K, N, long_groups, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    ends = ends_of(G, long_groups)
    rows = ends[-1] + 9  # the last rows belong to no group
    assert rows <= 128 * G  # the ring kernel's calls
    a = torch.randn(rows, K, generator=g, device=dev).bfloat16()
    w = torch.randn(G, N, K, generator=g, device=dev).bfloat16()
    return a, w, torch.tensor(ends, dtype=torch.int32, device=dev), ends


def groups(ends):
    return [(g, lo, hi) for g, (lo, hi) in enumerate(zip([0] + ends, ends)) if hi > lo]


@pytest.mark.parametrize("G,K,N", SHAPES)
@pytest.mark.parametrize("long_groups", [False, True])
def test_bf16(cuda, G, K, N, long_groups):
    print("runs bf16 G=%d K=%d N=%d long=%d" % (G, K, N, long_groups), flush=True)
    a, w, offs, ends = inputs(G, K, N, long_groups, cuda, K + N)
    out = torch.full((a.shape[0], N), 7.0, dtype=torch.bfloat16, device=cuda)
    M.grouped_gemm(a, w, offs, out=out)
    for g, lo, hi in groups(ends):
        ref = a[lo:hi].double() @ w[g].double().t()
        mag = a[lo:hi].double().abs() @ w[g].double().abs().t()
        err = (out[lo:hi].double() - ref).abs()
        assert bool((err <= ref.abs() * 2.0 ** -8 + K * 2.0 ** -24 * mag).all()), (g, lo, hi)
    assert bool((out[ends[-1]:] == 7.0).all())


@pytest.mark.parametrize("G,K,N", SHAPES)
@pytest.mark.parametrize("long_groups", [False, True])
def test_swiglu_rows(cuda, G, K, N, long_groups):
    """The same rows through a_rows, each group against the call that has it alone: one
    group of up to 128 rows is above the ring kernel's average, so its tile is the
    256-row loop's, with the same sums."""
    print("runs swiglu G=%d K=%d N=%d long=%d" % (G, K, N, long_groups), flush=True)
    a, w, offs, ends = inputs(G, K, N, long_groups, cuda, K * 3 + N)
    up = w.flip(0).contiguous()
    idx = torch.randperm(a.shape[0], device=cuda).int()
    out = torch.full((a.shape[0], N), 7.0, dtype=torch.bfloat16, device=cuda)
    M.grouped_swiglu(a, w, up, offs, a_rows=idx, out=out)
    for g, lo, hi in groups(ends)[::7] + groups(ends)[-2:]:
        rows = a[idx[lo:hi].long()]
        rows = torch.cat([rows, rows.new_zeros(129, K)])  # 129 rows or more in one group
        one = torch.tensor([rows.shape[0]], dtype=torch.int32, device=cuda)
        ref = M.grouped_swiglu(rows, w[g:g + 1].contiguous(), up[g:g + 1].contiguous(), one)
        assert torch.equal(out[lo:hi], ref[:hi - lo]), (g, lo, hi)
    assert bool((out[ends[-1]:] == 7.0).all())


@pytest.mark.parametrize("G,K,N", [s for s in SHAPES if s[1] % 128 == 0])
@pytest.mark.parametrize("long_groups", [False, True])
def test_int8(cuda, G, K, N, long_groups):
    print("runs int8 G=%d K=%d N=%d long=%d" % (G, K, N, long_groups), flush=True)
    a, w, offs, ends = inputs(G, K, N, long_groups, cuda, K * 5 + N)
    q, s = M.quant_rows_i8(a)
    wq, ws = M.quant_rows_i8(w)
    out = torch.full((a.shape[0], N), 7.0, dtype=torch.bfloat16, device=cuda)
    M.grouped_gemm_i8(q, s, wq, ws, offs, out=out)
    for g, lo, hi in groups(ends):
        acc = q[lo:hi].double() @ wq[g].double().t()  # exact integers
        ref = (acc.float() * (s[lo:hi, None] * ws[g][None])).bfloat16()
        assert torch.equal(out[lo:hi], ref), (g, lo, hi)
    assert bool((out[ends[-1]:] == 7.0).all())


@pytest.mark.parametrize("ident_m", [5, 128])
def test_identity_rows(cuda, ident_m):
    """Groups of ident_m rows read ident_a, also in runs."""
    G, K, N = 130, 128, 1288
    a, w, offs, ends = inputs(G, K, N, False, cuda, ident_m)
    ident = torch.randn(ident_m, K, device=cuda).bfloat16()
    out = M.grouped_gemm(a, w, offs, ident_a=ident, ident_m=ident_m)
    full = a.clone()
    for g, lo, hi in groups(ends):
        if hi - lo == ident_m:
            full[lo:hi] = ident
    assert torch.equal(out[:ends[-1]], M.grouped_gemm(full, w, offs)[:ends[-1]])
