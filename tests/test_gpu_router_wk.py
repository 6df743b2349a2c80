"""The router GEMM with K split over the waves of a block (csrc/router_wk.hip):
logits against the float64 product, at token counts on both sides of its tiles
(16 to 128 tokens) and of the rule that picks it, for bf16 and fp32 weights.

Bound: a sum of H products in fp32 in any order is within H * 2^-24 * sum |x||w|;
an fp32 weight's hi/lo split adds 2^-16 of that sum (hi + lo keeps 16 bits of w)."""
import pytest
import torch

import moe_route as M
from moe_route.configs import RouteCfg

pytestmark = pytest.mark.gpu

# (E, H): H = 64 leaves three of the four waves without a K step, 576 splits
# unevenly, the rest are the fused kernel's shapes and ordinary ones
SHAPES = [(32, 64), (64, 576), (128, 2048), (256, 7168), (256, 1024)]
TOKENS = [1, 15, 17, 48, 257, 513, 1025, 3073, 4133, 6001]


def inputs(T, H, E, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(T, H, generator=g, device=dev).bfloat16()
    return x, torch.randn(E, H, generator=g, device=dev) * 0.02


def assert_logits(got, x, w, split):
    ref = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    bound = (2 * x.shape[1] * 2.0 ** -24 + (2.0 ** -16 if split else 0.0)) * mag
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("E,H", SHAPES)
@pytest.mark.parametrize("T", TOKENS)
@pytest.mark.parametrize("fp32", [False, True])
def test_logits(cuda, E, H, T, fp32):
    print("router_wk E=%d H=%d T=%d fp32=%d" % (E, H, T, fp32), flush=True)
    x, w = inputs(T, H, E, T + E, cuda)
    w = w if fp32 else w.bfloat16()
    k = min(8, E)
    logits, ids, wts, counts = M.route(x, w, None, k, RouteCfg())
    assert_logits(logits, x, w, fp32)
    # the scoring on the same logits, and the histogram
    i2, w2, c2 = M.topk(logits, None, k, RouteCfg())
    assert torch.equal(ids, i2) and torch.equal(wts, w2) and torch.equal(counts, c2)
    if not fp32:
        assert_logits(M.router_gemm(x, w), x, w, False)


# (E, H, T): the 128 x 64 tiles with 41, 81, 82 and 127 row tiles (the grid rounds them up
# to a multiple of 8), the 128 x 128 tiles, and E = 128 either side of each line of the rule
LARGE = [(256, 1024, 5121), (256, 4096, 8065), (128, 1024, 10241), (128, 1024, 10369),
         (128, 1024, 16256), (256, 1024, 8193), (256, 1024, 12001), (128, 8192, 16385),
         (128, 1024, 10240), (128, 4096, 10241), (128, 1024, 16385), (128, 8192, 32769)]


@pytest.mark.parametrize("E,H,T", LARGE)
def test_large_batches(cuda, E, H, T):
    print("router_wk large E=%d H=%d T=%d" % (E, H, T), flush=True)
    x, w = inputs(T, H, E, T + H, cuda)
    w = w.bfloat16()
    logits, ids, wts, counts = M.route(x, w, None, 8, RouteCfg())
    for lo in range(0, T, 8192):  # the float64 copies a piece at a time
        assert_logits(logits[lo:lo + 8192], x[lo:lo + 8192], w, False)
    i2, w2, c2 = M.topk(logits, None, 8, RouteCfg())
    assert torch.equal(ids, i2) and torch.equal(wts, w2) and torch.equal(counts, c2)


def test_unaligned_logits(cuda):
    """moe_router_gemm takes logits at any 4-byte address."""
    T, H, E = 33, 1024, 64
    x, w = inputs(T, H, E, 5, cuda)
    w = w.bfloat16()
    buf = torch.full((T * E + 2,), -7.0, device=cuda)
    out = buf[1:-1]
    M._check(M.lib().moe_router_gemm(M._ptr(x), M._ptr(w), T, H, E, M._ptr(out), M._stream(x)))
    assert torch.equal(out.view(T, E), M.router_gemm(x, w))
    assert float(buf[0]) == -7.0 and float(buf[-1]) == -7.0


@pytest.mark.parametrize("E,H,T", [(256, 7168, 16384), (256, 7168, 16385), (256, 7168, 16500),
                                   (128, 2048, 10240), (128, 2048, 10241), (128, 2048, 10370)])
@pytest.mark.parametrize("rule", ["sigmoid_group", "softmax", "softmax_bias"])
def test_fused_kernel_either_side_of_the_rule(cuda, E, H, T, rule):
    """At the fused kernel's shapes: the last batch that goes to this GEMM, the
    first that goes to the fused kernel, and one that ends inside a fused tile;
    logits, ids, weights and counts equal the standalone GEMM and scoring."""
    cfg = {"sigmoid_group": RouteCfg(M.SCORING_SIGMOID_GROUP, True, E // 32, 4, 2.5),
           "softmax": RouteCfg(M.SCORING_SOFTMAX, True),
           "softmax_bias": RouteCfg(M.SCORING_SOFTMAX_BIAS, True, norm_min=1e-6)}[rule]
    k = 8 if T % 2 else 5
    x, w = inputs(T, H, E, T, cuda)
    w = w.bfloat16()
    bias = torch.randn(E, device=cuda, generator=torch.Generator(device=cuda).manual_seed(T)) * 0.1
    logits, ids, wts, counts = M.route(x, w, bias, k, cfg)
    assert torch.equal(logits, M.router_gemm(x, w))
    i2, w2, c2 = M.topk(logits, bias, k, cfg)
    assert torch.equal(ids, i2) and torch.equal(wts, w2) and torch.equal(counts, c2)


@pytest.mark.parametrize("topk_group", [1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("k", [8, 6])
def test_fused_kernel_ties(cuda, topk_group, k):
    """The fused kernel's epilogue ranks two tokens per lane group (with at most 4
    kept groups in compacted rounds): the same choice as the scoring kernel where
    scores tie exactly inside and across groups (rows and bias repeat every 37)."""
    E, H, T = 256, 7168, 16391
    cfg = RouteCfg(M.SCORING_SIGMOID_GROUP, True, 8, topk_group, 2.5)
    x, w = inputs(T, H, 37, 100 + topk_group, cuda)
    at = torch.arange(E, device=cuda) % 37
    w = w.bfloat16()[at].contiguous()
    bias = (torch.arange(37, device=cuda) * 0.37).sin()[at].contiguous()
    logits, ids, wts, counts = M.route(x, w, bias, k, cfg)
    assert torch.equal(logits[:, 0], logits[:, 37])
    i2, w2, c2 = M.topk(logits, bias, k, cfg)
    assert torch.equal(ids, i2) and torch.equal(wts, w2) and torch.equal(counts, c2)


@pytest.mark.parametrize("E,H,T,k", [(256, 7168, 16391, 8), (256, 7168, 16391, 2),
                                     (128, 2048, 10241, 8), (128, 2048, 10241, 4)])
def test_fused_kernel_block_histograms(cuda, E, H, T, k):
    """The fused kernel's histogram handoff in the one-call step: the same
    permutation as from the ids alone."""
    x, w = inputs(T, H, E, T + k, cuda)
    w = w.bfloat16()
    plan = M.MoePlan(T, H, E, k, RouteCfg(), cuda)
    plan.route_permute(x, w, None, index_only=True)
    p = M.permute(x, plan.topk_ids, E, index_only=True)
    for name in ("row_token", "pair_row", "offsets", "counts"):
        assert torch.equal(getattr(plan, name), p[name]), name


# (E, H, T, fp32, parts): shapes outside the rule whose K is split over blocks into parts of
# unequal length, and three whose H is an odd number of 64s and stays whole
PARTS = [(64, 8192, 4133, True, 3), (64, 8192, 4904, True, 3), (256, 8192, 4133, False, 7),
         (128, 4608, 6001, True, 5), (256, 1024, 2100, True, 7), (256, 8704, 5000, False, 6),
         (256, 8256, 5000, False, 1), (128, 4160, 6001, True, 1), (256, 1088, 1100, True, 1)]


def partitions(T, H, N):
    """The general GEMM's: doubled up to 8 while its tiles leave CUs idle and H divides
    (the workspace's count), then the largest whose rounds of 256 blocks are shortest."""
    bm, bn = (256, 128) if N >= 256 else (64, N)
    blocks, most = -(-T // bm) * -(-N // bn), 1
    while blocks * most < 256 and most < 8 and H % (128 * most) == 0:
        most *= 2
    return most, min(range(most, 0, -1), key=lambda p: -(-blocks * p // 256) / p)


@pytest.mark.parametrize("E,H,T,fp32,parts", PARTS)
def test_uneven_k_partitions(cuda, E, H, T, fp32, parts):
    """K split over blocks, the partial sums added by the scoring kernel."""
    N = 2 * E if fp32 else E
    most, run = partitions(T, H, N)
    assert run == parts and (parts == 1 or H // 64 % parts)
    sums = T * most * N * 4 if most * N > E else 0
    assert M.lib().moe_route_workspace_bytes(T, H, E, int(fp32)) == \
        (N * H * 2 if fp32 else 0) + (sums + 255) // 256 * 256
    x, w = inputs(T, H, E, T + E, cuda)
    w = w if fp32 else w.bfloat16()
    logits, ids, wts, counts = M.route(x, w, None, 8, RouteCfg())
    assert_logits(logits, x, w, fp32)
    i2, w2, c2 = M.topk(logits, None, 8, RouteCfg())
    assert torch.equal(ids, i2) and torch.equal(wts, w2) and torch.equal(counts, c2)


def chained(x, w, parts):
    """x . w^T as the matrix instruction adds it, a rounding to fp32 every 8 products, in
    `parts` chains of equal length that are then added."""
    x, w, U = x.double(), w.double(), x.shape[1] // 64
    total = None
    for z in range(parts):
        acc = None
        for k in range(z * U // parts * 64, (z + 1) * U // parts * 64, 8):
            p = x[:, k:k + 8] @ w[:, k:k + 8].t()
            acc = (p if acc is None else acc.double() + p).float()
        total = acc if total is None else total + acc
    return total


@pytest.mark.parametrize("E,H,T,parts", [
    (64, 4096, 128, 8), (64, 8192, 700, 8), (32, 1024, 2500, 8), (256, 2048, 1100, 8),  # waves
    (256, 4096, 8000, 4), (256, 1024, 12000, 4), (128, 1024, 12000, 2),  # whole-K tiles
    (256, 8192, 4904, 8), (128, 8192, 3000, 8)])  # fewer partitions than that
def test_error_of_the_sum(cuda, E, H, T, parts):
    """No further from the float64 product than K in as many fp32 chains as the general
    GEMM has partitions at this size.  3%: the two errors are norms over 8192 values and
    more, each within 1 / sqrt(2 * 8192) = 0.8% of its expectation."""
    x, w = inputs(T, H, E, 7, cuda)
    w = w.bfloat16()
    logits = M.route(x, w, None, 8, RouteCfg())[0]
    ref = x.double() @ w.double().t()
    err = float((logits.double() - ref).norm() / ref.norm())
    of_chains = float((chained(x, w, parts).double() - ref).norm() / ref.norm())
    print("sum E=%d H=%d T=%d: %.3g, %d chains %.3g" % (E, H, T, err, parts, of_chains), flush=True)
    assert err <= 1.03 * of_chains
