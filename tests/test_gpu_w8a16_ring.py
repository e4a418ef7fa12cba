"""The large-tile W8A16 kernels convert a step's weight codes during the step before, out of a register ring of two steps, or
of four under a long reduction: reductions shorter than the ring, reductions that end inside it, both sides of the rule
between the two, and experts whose rows fill a part of the tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# tokens x (H, I, E, K): 128- and 192-row tiles; a step is 64 elements, so H and I give 2, 4, 6, 10 and 16 steps, all in a
# ring of two, and 36, 38, 40, 42, 44 and 48: a ring of four from 40 on where it divides the steps and a tile holds more than
# 32 rows
@pytest.mark.parametrize("T,H,I,E,K", [
    (200, 128, 128, 4, 1), (200, 384, 128, 4, 1), (160, 640, 384, 4, 2), (330, 128, 640, 4, 2), (700, 384, 256, 4, 2),
    (333, 1024, 640, 8, 2), (200, 2560, 2688, 4, 1), (330, 2816, 2304, 4, 2), (700, 2432, 3072, 4, 2),
])
def test_codes_converted_a_step_ahead(pkg, dev, T, H, I, E, K):
    assert pkg.tile_rows(T, K, E) in (128, 192)
    g = torch.Generator().manual_seed(T + H + I)
    w13 = (torch.randn(E, 2 * I, H, generator=g) * 0.1).to(torch.float8_e4m3fn).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.1).to(torch.float8_e4m3fn).to(dev)
    s13 = torch.rand(E, 2 * I // 128, H // 128, generator=g).to(dev) + 0.5
    s2 = torch.rand(E, H // 128, I // 128, generator=g).to(dev) + 0.5
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    # the first experts take most tokens, the last one a handful: full tiles, part tiles and one m-tile
    score = torch.rand(T, E, generator=g) + torch.arange(E, 0, -1) * 0.35
    score[5:, E - 1] = -1.0
    ids = score.topk(K, dim=1).indices.to(torch.int32).to(dev)
    got = pkg.fused_experts_w8a16(x, pkg.pack_weights(w13), s13, pkg.pack_weights(w2), s2, ids)
    # the bf16 kernels on bf16(code * scale): the same products, summed in another order inside the matrix instruction
    deq = lambda q, s: (q.float() * s.repeat_interleave(128, 1).repeat_interleave(128, 2)).to(torch.bfloat16)
    want = pkg.fused_experts_bf16(x, pkg.pack_weights(deq(w13, s13)), pkg.pack_weights(deq(w2, s2)), ids)
    gf, wf = got.float(), want.float()
    # a neighbouring bf16 (2^-7 of the value) in the intermediate or the result, and its echo in sums that cancel
    assert ((gf - wf).abs() <= 1.6e-2 * wf.abs() + 2e-3 * wf.pow(2).mean().sqrt()).all()
    assert (got.view(torch.int16) == want.view(torch.int16)).float().mean().item() >= 0.97


@pytest.mark.parametrize("M,K,N", [(100, 128, 128), (100, 384, 128), (100, 640, 272), (3000, 1408, 4096), (100, 512, 128)])
def test_an_infinite_activation_in_the_last_step_stays_infinite(pkg, dev, M, K, N):
    """128- and 192-row tiles, an odd number of 128-blocks (and an even one): no step past the reduction's end touches the
    last token tile.  Against the de-quantised operands' product in 64 bits: the same elements are +Inf, -Inf and NaN (an
    infinity against a zero code), every other row is finite."""
    g = torch.Generator().manual_seed(M + K)
    w = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
    s = torch.rand(-(-N // 128), K // 128, generator=g) + 0.5
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    cols = {3: K - 1, 40: K - 64, M - 1: K - 33, 17: 5}
    for row, col in cols.items():
        x[row, col] = float("inf") if col % 2 else float("-inf")
    got = pkg.mm_w8a16(x.to(dev), pkg.pack_weights(w.to(dev)), s.to(dev)).float().cpu()
    rows = list(cols)
    wd = w.double() * s.double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
    want = x[rows].double() @ wd.t()
    assert torch.equal(got[rows].isnan(), want.isnan())
    assert torch.equal(got[rows].isposinf(), want.isposinf()) and torch.equal(got[rows].isneginf(), want.isneginf())
    assert got[[i for i in range(M) if i not in cols]].isfinite().all()
