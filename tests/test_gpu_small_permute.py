"""The permute of a small batch (index pass and gather in one launch) against the
general index kernels (an index-only permute) and the rows they name: pair counts
at its limits (2048; 1024 for the shortest rows), rows of one and of several blocks,
one to 1024 experts, invalid ids, and every k with its own instantiation."""
import pytest
import torch

import moe_route as M

pytestmark = pytest.mark.gpu

CASES = [
    # (T, k, E, H, x dtype, fp8)
    (1, 1, 1, 512, torch.bfloat16, False),
    (1, 8, 256, 7168, torch.bfloat16, False),
    (128, 8, 64, 512, torch.bfloat16, False),    # 1024 pairs of 64-item rows: the last
    (129, 8, 64, 512, torch.bfloat16, False),    # one too many: the general path
    (256, 8, 256, 1032, torch.bfloat16, False),  # 2048 pairs, 129 items a row
    (257, 8, 256, 1032, torch.bfloat16, False),  # general path
    (256, 4, 32, 1024, torch.bfloat16, False),   # 1024 pairs: 4 ids a thread
    (205, 5, 64, 1032, torch.bfloat16, False),   # 1025: 8
    (513, 2, 8, 2048, torch.bfloat16, True),
    (682, 3, 1024, 1024, torch.bfloat16, False),
    (1023, 2, 8, 1160, torch.bfloat16, False),
    (100, 6, 40, 260, torch.float32, False),     # 65 items a row
    (16, 8, 256, 7168, torch.bfloat16, True),
    (256, 8, 128, 2048, torch.bfloat16, True),   # 2048 pairs, 128 items a row
    (333, 3, 7, 1152, torch.bfloat16, True),     # 72 items a row, 999 pairs
    (77, 2, 8, 4096, torch.bfloat16, True),
]


@pytest.mark.parametrize("T,k,E,H,dtype,fp8", CASES)
@pytest.mark.parametrize("invalid", [False, True])
def test_small_permute(cuda, T, k, E, H, dtype, fp8, invalid):
    print("small permute T=%d k=%d E=%d H=%d fp8=%d" % (T, k, E, H, fp8), flush=True)
    g = torch.Generator(device=cuda).manual_seed(T * 7 + E)
    x = torch.randn(T, H, generator=g, device=cuda).to(dtype)
    ids = torch.randint(0, E, (T, k), generator=g, device=cuda, dtype=torch.int32)
    if invalid:
        drop = torch.rand(T, k, generator=g, device=cuda) < 0.3
        bad = torch.where(torch.rand(T, k, generator=g, device=cuda) < 0.5, -1, E + 5).int()
        ids = torch.where(drop, bad, ids).contiguous()
    p = M.permute(x, ids, E, fp8=fp8)
    ref = M.permute(x, ids, E, index_only=True)
    assert torch.equal(p["pair_row"], ref["pair_row"])
    assert torch.equal(p["offsets"], ref["offsets"]) and torch.equal(p["counts"], ref["counts"])
    rows = int(ref["offsets"][-1])
    assert rows == int(((ids >= 0) & (ids < E)).sum())
    rt = ref["row_token"][:rows].long()
    assert torch.equal(p["row_token"][:rows], ref["row_token"][:rows])
    if not fp8:
        assert torch.equal(p["xg"][:rows], x[rt])
        return
    # one token to one expert gives the token's own bytes and scales
    one = M.permute(x, torch.zeros(T, 1, dtype=torch.int32, device=cuda), 1, fp8=True)
    assert torch.equal(p["xg"][:rows], one["xg"][rt])
    assert torch.equal(p["scales"][:rows], one["scales"][rt])
