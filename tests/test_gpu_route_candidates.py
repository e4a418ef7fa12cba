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


# every road of the selection: one token to a workgroup, one to a wavefront, groups of 32 and others
@pytest.mark.parametrize("T", [7, 96])
@pytest.mark.parametrize("E,K,n_groups,topk_groups", [(8, 2, 1, 1), (128, 8, 1, 1), (256, 8, 8, 4), (60, 7, 12, 5), (249, 8, 3, 2), (300, 8, 1, 1)])
def test_nan_scores_come_first_whatever_the_batch(pkg, oracle, dev, T, E, K, n_groups, topk_groups):
    """NaN of either sign before everything else, lower index first, in a row and among the groups' sums: the oracle's order
    (torch.sort), on every road."""
    g = torch.Generator().manual_seed(E + T)
    x = torch.randn(T, E, generator=g)
    both = torch.tensor([0x7fc00000, 0xffc00000 - 2 ** 32], dtype=torch.int32).view(torch.float32)
    where = torch.rand(T, E, generator=g) < 0.02
    x[where] = both[torch.randint(0, 2, (int(where.sum()),), generator=g)]
    x[1] = both[1]                                        # nothing but NaN
    x[2, : E // n_groups] = both[0]                       # a whole group (or everything)
    x[3] = float("-inf")
    x[3, E // 2] = both[1]
    x[4, 0], x[4, 1:E // n_groups] = float("inf"), float("-inf")         # a group whose sum is NaN
    want, want_ids = oracle.select_sigmoid_grouped(x, None, K, n_groups, topk_groups, scale=1.0, renorm=False)
    w, ids = pkg.moe_route(x.to(dev), K, "scores", None, n_groups, topk_groups, renorm=False)
    assert torch.equal(ids.cpu(), want_ids)
    torch.testing.assert_close(w.cpu(), want, rtol=0, atol=0, equal_nan=True)
    if n_groups > 1:
        values, idx = torch.empty(T, K, device=dev), torch.empty(T, K, dtype=torch.int32, device=dev)
        pkg.noaux_tc_topk(values, idx, x.to(dev), n_groups, topk_groups, K)
        assert torch.equal(idx.cpu(), want_ids)


@pytest.mark.parametrize("E,K,n_groups,topk_groups", [(256, 8, 8, 4), (256, 32, 8, 1), (256, 32, 8, 7), (128, 6, 64, 3), (249, 8, 3, 2), (4, 2, 2, 1)])
def test_fewer_finite_scores_than_picks_under_a_group_limit(pkg, oracle, dev, E, K, n_groups, topk_groups):
    """Row t has t finite scores, from none to more than K: the rest of the picks are -inf ones, lowest index first, of kept and
    dropped groups alike."""
    g = torch.Generator().manual_seed(E + K)
    T = min(K + 3, E)
    x = torch.full((T, E), float("-inf"))
    for t in range(T):
        x[t, torch.randperm(E, generator=g)[:t]] = torch.randn(t, generator=g)
    _, want_ids = oracle.select_sigmoid_grouped(x, None, K, n_groups, topk_groups, renorm=False)
    for rows in (x, x.repeat(65 // T + 1, 1)):            # a workgroup per token, and more than 64 tokens
        _, ids = pkg.moe_route(rows.to(dev), K, "scores", None, n_groups, topk_groups, renorm=False)
        assert torch.equal(ids[:T].cpu(), want_ids) and torch.equal(ids[-T:].cpu(), want_ids)
