"""The permutation in one launch (257 to 16384 slots) at the edges of its range and of its chunks, against the oracle's counting
sort: every slot's row, the experts' offsets, and - through the experts' op, which reads it - the tile list."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DIRECT_SLOTS = 16384


def _ids(T, K, E, seed, dropped=0.0):
    g = torch.Generator().manual_seed(seed)
    ids = torch.argsort(torch.rand(T, E, generator=g), dim=-1)[:, :K].to(torch.int32)
    if dropped:
        out = torch.rand(T, K, generator=g) < dropped
        ids[out] = torch.where(torch.rand(int(out.sum()), generator=g) < 0.5, torch.tensor(-1), torch.tensor(E)).to(torch.int32)
    return ids


@pytest.mark.parametrize("T,K,E,dropped", [
    (257, 1, 1, 0.0), (257, 1, 2, 0.3), (129, 2, 3, 0.0), (511, 1, 64, 0.0), (64, 8, 65, 0.1), (300, 8, 128, 0.0),
    (1023, 5, 257, 0.0), (DIRECT_SLOTS // 8 - 1, 8, 256, 0.05), (DIRECT_SLOTS // 8, 8, 1024, 0.0),
    (DIRECT_SLOTS // 8 + 1, 8, 1024, 0.0), (DIRECT_SLOTS, 1, 8, 0.0), (DIRECT_SLOTS + 1, 1, 8, 0.02),
])
def test_rows_and_offsets_are_the_stable_sort(pkg, dev, T, K, E, dropped):
    ids = _ids(T, K, E, 7 * T + E, dropped)
    ss, off, s2r = (t.cpu() for t in pkg.moe_permute(ids.to(dev), E))
    flat = ids.flatten().long()
    valid = (flat >= 0) & (flat < E)
    n = int(valid.sum())
    want = torch.sort(torch.where(valid, flat, E), stable=True).indices[:n]
    assert torch.equal(ss[:n].long(), want)
    rows = torch.full((T * K,), -1)
    rows[want] = torch.arange(n)
    assert torch.equal(s2r.long(), rows)
    counts = torch.bincount(flat[valid], minlength=E)
    assert torch.equal(off.long(), torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]))


def test_ids_that_start_off_a_sixteen_byte_boundary(pkg, dev):
    T, K, E = 401, 3, 40
    ids = _ids(T, K, E, 5)
    room = torch.empty(T * K + 1, dtype=torch.int32, device=dev)
    view = room[1:].view(T, K)
    view.copy_(ids)
    for got, want in zip(pkg.moe_permute(view, E), pkg.moe_permute(ids.to(dev), E)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("T", [DIRECT_SLOTS // 4, DIRECT_SLOTS // 4 + 1])
def test_one_hot_expert_and_empty_ones_reach_the_gemms(pkg, oracle, dev, T):
    """One expert holds a row of every token (dozens of row tiles), half of the others none: rows of a batch on either side of
    the limit equal, bit for bit, the same tokens' rows in small batches."""
    H, I, E, K = 256, 128, 16, 4
    ld = pkg.pack_layer(*(t.to(dev) for t in oracle.make_layer(E, H, I, seed=3)))
    g = torch.Generator().manual_seed(T)
    ids = torch.stack([torch.cat([torch.tensor([5]), 8 + torch.randperm(8, generator=g)[:K - 1]]) for _ in range(T)]).to(torch.int32).to(dev)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    big = pkg.fused_experts_fp8(x, *ld, ids)
    for lo in (0, T // 2, T - 40):
        assert torch.equal(big[lo:lo + 40], pkg.fused_experts_fp8(x[lo:lo + 40].contiguous(), *ld, ids[lo:lo + 40].contiguous()))


# one and two picks, chunks on either side of the line from which counts are kept in copies, experts at the edges of 8, 4, 2 and 1
@pytest.mark.parametrize("T,K,E", [(6144, 1, 8), (6145, 1, 8), (DIRECT_SLOTS, 1, 1), (DIRECT_SLOTS, 1, 128), (DIRECT_SLOTS, 1, 129), (16001, 1, 256),
                                   (DIRECT_SLOTS, 1, 257), (DIRECT_SLOTS, 1, 512), (12345, 1, 513), (DIRECT_SLOTS // 2, 2, 2), (8111, 2, 64), (6144, 2, 8), (6145, 2, 8),
                                   (DIRECT_SLOTS // 2, 2, 65)])
@pytest.mark.parametrize("load", ["even", "collapsed", "half outside"])
def test_counts_kept_in_copies_add_up(pkg, dev, T, K, E, load):
    ids = _ids(T, K, E, T + E, 0.5 if load == "half outside" else 0.0)
    if load == "collapsed":
        ids[:] = torch.arange(E - K, E, dtype=torch.int32)
    ss, off, s2r = (t.cpu() for t in pkg.moe_permute(ids.to(dev), E))
    flat = ids.flatten().long()
    valid = (flat >= 0) & (flat < E)
    n = int(valid.sum())
    want = torch.sort(torch.where(valid, flat, E), stable=True).indices[:n]
    rows = torch.full((T * K,), -1)
    rows[want] = torch.arange(n)
    assert torch.equal(ss[:n].long(), want) and torch.equal(s2r.long(), rows)
    counts = torch.bincount(flat[valid], minlength=E)
    assert torch.equal(off.long(), torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]))
