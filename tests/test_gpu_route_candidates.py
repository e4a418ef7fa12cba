"""The one-token routing workgroup compares the best of every part of the row: against the per-wavefront kernel, which looks
at the whole row, on the same rows (a batch of more than 64 tokens runs that one)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# parts of 64 experts (one short of, exactly, one past a wavefront) and groups: even, odd and two-wide ones, as many picks as a
# group, as the kept groups hold, as there are experts
@pytest.mark.parametrize("E,K,n_groups,topk_groups", [
    (8, 2, 1, 1), (8, 8, 1, 1), (63, 8, 1, 1), (64, 32, 1, 1), (65, 8, 1, 1), (128, 8, 1, 1), (200, 32, 1, 1), (256, 1, 1, 1),
    (256, 8, 8, 4), (256, 32, 8, 1), (256, 32, 8, 2), (128, 6, 64, 3), (249, 8, 3, 2), (60, 7, 12, 12), (256, 8, 4, 4)])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "scores"])
def test_picks_of_one_token_equal_the_whole_rows(pkg, dev, E, K, n_groups, topk_groups, mode):
    g = torch.Generator().manual_seed(E * 64 + K)
    x = torch.randn(96, E, generator=g)
    x[1::8] = x[1::8].round()                             # many equal scores
    x[2::8] = 0.0                                         # all equal, of both signs of zero
    x[2::8, ::2] *= -1.0
    bias = None
    if mode != "softmax":
        bias = torch.randn(E, generator=g)
        bias[torch.randperm(E, generator=g)[:E // 3]] = float("-inf")          # picks that are no better than a dropped group
        if mode == "scores":
            x[3::8, : E - 1] = float("-inf")
        bias = bias.to(dev)
    x = x.to(dev)
    args = (K, mode, bias, n_groups, topk_groups)
    w_all, ids_all = pkg.moe_route(x, *args)
    for t0 in (0, 8):
        w, ids = pkg.moe_route(x[t0:t0 + 8].contiguous(), *args)
        assert torch.equal(ids, ids_all[t0:t0 + 8])
        assert torch.equal(w.view(torch.int32), w_all[t0:t0 + 8].view(torch.int32))
