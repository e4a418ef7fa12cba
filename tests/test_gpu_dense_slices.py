"""Dense FP8 products whose reduction is cut into slices, on the grouped kernel (every tile height, the last slice as long as
the others, shorter, a single step) and on the kernels of few rows, against the quantised operands' product in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# what the shape is to run: kernel, token rows of a work item, slices, steps of the last slice
@pytest.mark.parametrize("M,K,N,plan", [
    (33, 18432, 7168, ("sliced", 64, 9, 16)), (64, 16512, 4096, ("sliced", 64, 9, 1)), (50, 18560, 7168, ("sliced", 64, 5, 17)),
    (64, 32768, 1024, ("sliced", 64, 16, 16)),
    (150, 14336, 4096, ("sliced", 128, 7, 16)), (300, 18432, 7168, ("sliced", 128, 3, 48)), (520, 16512, 1024, ("sliced", 128, 9, 1)),
    (300, 18560, 7168, ("sliced", 128, 3, 17)), (1000, 16640, 1040, ("sliced", 128, 5, 2)), (200, 16896, 4096, ("sliced", 128, 5, 4)),
    (1501, 16384, 1008, ("sliced", 128, 4, 32)), (128, 18432, 272, ("sliced", 128, 9, 16)), (600, 8320, 272, ("sliced", 128, 5, 1)),
    (520, 16384, 1024, ("sliced", 128, 8, 16)), (700, 16384, 1040, ("sliced", 128, 8, 16)),
    (129, 18432, 7168, ("sliced", 192, 9, 16)), (150, 18560, 4096, ("sliced", 192, 10, 1)),
    # a workgroup per 16 columns: 1, 2 and 4 row tiles, columns past the last eight, slices that end inside a batch of steps
    (1, 7168, 1536, ("narrow", 16, 1, 56)), (16, 2176, 1040, ("narrow", 16, 1, 17)), (32, 7168, 2048, ("narrow", 16, 1, 56)),
    (64, 16384, 1024, ("narrow", 16, 1, 128)), (32, 18432, 1024, ("narrow", 16, 1, 144)), (17, 16384, 16, ("narrow", 16, 1, 128)),
    (31, 2304, 4096, ("narrow", 32, 1, 18)), (17, 4736, 4096, ("narrow", 32, 1, 37)), (33, 4096, 2064, ("narrow", 64, 1, 32)),
    # a wavefront per work item
    (17, 18432, 16, ("wavefront", 32, 36, 4)), (64, 7168, 4096, ("wavefront", 64, 14, 4)), (64, 7168, 4112, ("wavefront", 64, 7, 8)),
    (385, 4736, 272, ("wavefront", 64, 10, 1)), (417, 8320, 16, ("wavefront", 64, 17, 1))])
def test_sliced_product(pkg, dev, M, K, N, plan):
    kernel, rows, slices, steps = pkg.ops.mm_plan(M, K, N)
    assert (kernel, rows, slices, K // 128 - (slices - 1) * steps) == plan
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(dev)
    ws = (torch.rand(-(-N // 128), K // 128, generator=g) + 0.5).to(dev)
    out = pkg.mm_fp8(x, pkg.pack_weights(w), ws)
    q, s = pkg.act_quant(x)
    xd = (q.double().view(M, K // 128, 128) * s[:, :K // 128, None].double()).view(M, K)
    wd = w.double() * ws.double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
    want = xd @ wd.t()
    d = (out.double() - want).abs()
    # bf16 result: half a unit in the last place, 2^-9 of the value; the matrix instruction's internal error (2^-11.8 of
    # the largest of 128 products, 4.5 times an element's size squared) adds about 1e-3 of the result's spread
    assert (d <= 2.0 ** -8 * want.abs() + 4e-3 * want.pow(2).mean().sqrt()).all(), d.max().item()
    assert torch.equal(out.view(torch.int16), pkg.mm_fp8(x, pkg.pack_weights(w), ws).view(torch.int16))


# strips of 128 columns: whole under 128- and 192-row tiles, and slices; a last row tile of one m-tile (its second wavefront
# of a pair has none), of one row, whole; columns that end inside a strip; an odd number of steps; exactly one round of items
@pytest.mark.parametrize("M,K,N,plan", [
    (300, 7168, 7168, ("grouped", 128, 1, 56)), (385, 2176, 7152, ("grouped", 128, 1, 17)), (1040, 2048, 2000, ("grouped", 128, 1, 16)),
    (2048, 4096, 2048, ("grouped", 128, 1, 32)), (140, 4096, 28672, ("grouped", 192, 1, 32)), (155, 4224, 28672, ("grouped", 192, 1, 33)),
    (400, 7168, 1536, ("sliced", 128, 4, 8)), (560, 7296, 1520, ("sliced", 128, 4, 9)), (200, 7168, 2112, ("sliced", 128, 4, 8))])
def test_strips_of_128_columns(pkg, dev, M, K, N, plan):
    test_sliced_product(pkg, dev, M, K, N, plan)


@pytest.mark.parametrize("M,K,N", [(300, 7168, 7168), (385, 2176, 7152), (155, 4224, 28672)])
def test_whole_products_in_strips_of_128_columns_keep_every_sum(pkg, dev, M, K, N):
    """The rows' bits are those of a batch that takes the wide strips; an infinity in the last step adds no NaN."""
    g = torch.Generator().manual_seed(M + K)
    w, ws = (t[0] for t in pkg.synthetic_weights(1, -(-N // 128) * 128, K, dev, 5))
    w, n = w[:N].contiguous(), -(-N // 128)
    x = torch.randn(4096, K, generator=g).to(torch.bfloat16).to(dev)
    got = pkg.mm_fp8(x[:M].contiguous(), w, ws[:n])
    assert torch.equal(got, pkg.mm_fp8(x, w, ws[:n])[:M])
    xi = x[:M].clone()
    xi[M - 1, K - 1] = float("inf")
    inf = pkg.mm_fp8(xi, w, ws[:n])
    assert torch.equal(inf[:M - 1], got[:M - 1]) and not inf[M - 1].isnan().all()


@pytest.mark.parametrize("M,H,I", [(33, 1024, 12288), (64, 256, 12416), (65, 512, 8192), (128, 1024, 18432), (257, 512, 9216)])
def test_gated_mlp_of_few_rows_on_the_grouped_kernels(pkg, dev, M, H, I):
    """Against the same layer run row block by row block on the per-wavefront kernels (at most 32 rows)."""
    w13, s13 = (t[0] for t in pkg.synthetic_weights(1, 2 * I, H, dev, 3))
    w2, s2 = (t[0] for t in pkg.synthetic_weights(1, H, I, dev, 4))
    x = torch.randn(M, H, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(dev)
    got = pkg.mlp_fp8(x, w13, s13, w2, s2).float()
    want = torch.cat([pkg.mlp_fp8(x[i:i + 32].contiguous(), w13, s13, w2, s2) for i in range(0, M, 32)]).float()
    # the first product's sums are formed in another order: an element of the intermediate on a rounding boundary takes
    # the neighbouring e4m3 code (up to 1/8 of its value) in about 0.2 % of the elements, sqrt(0.002) / 8 / sqrt(3) = 0.003
    # of the result's spread, 0.02 at seven standard deviations; bf16 adds 2^-8 of the value
    d = (got - want).abs()
    rms = want.pow(2).mean().sqrt()
    assert (d <= 2.0 ** -7 * want.abs() + 0.02 * rms).all() and d.pow(2).mean().sqrt() <= 0.006 * rms


# reductions that end inside a batch of steps: per-wavefront kernels (four and two steps a batch), sliced products on the tall
# tiles with an odd number of steps in the last slice
@pytest.mark.parametrize("M,K,N", [(1, 2304, 256), (1, 4096, 256), (1, 14336, 256), (16, 5120, 1024), (32, 2304, 256),
                                   (64, 18048, 128), (520, 16512, 1024), (150, 18560, 4096)])
def test_an_infinite_scale_in_the_last_step_adds_no_nan(pkg, dev, M, K, N):
    """The quantised operands' product, group by group, in 64 bits: an activation group whose scale is infinite gives
    infinities of the same signs, not the NaN of a step past the end that counts it times zero."""
    g = torch.Generator().manual_seed(M + K)
    w = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(dev)
    ws = (torch.rand(-(-N // 128), K // 128, generator=g) + 0.5).to(dev)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    rows = sorted({0, M // 2, M - 1})
    cols = [K - 1, K // 2 + 3, 128 * (K // 2048) + 383]
    for i, col in enumerate(cols):                        # one infinity in a row; with one row, one call for each
        for row in rows[i:i + 1] if M > 1 else [0]:
            xi = x.clone()
            xi[row, col] = float("inf")
            xi = xi.to(dev)
            got = pkg.mm_fp8(xi, pkg.pack_weights(w), ws)[row].float()
            q, s = pkg.act_quant(xi[row:row + 1])
            p = (q.double().view(K // 128, 1, 128) @ w.double().view(N, K // 128, 128).permute(1, 2, 0)).squeeze(1)
            want = (p * (s[0, :K // 128, None].double() * ws.double().repeat_interleave(128, 0)[:N].t())).sum(0)
            assert torch.equal(got.isnan(), want.isnan()), (row, col, got.isnan().sum().item(), want.isnan().sum().item())
            assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())


def test_one_workspace_made_for_the_largest_batch_serves_the_smaller_ones(pkg, dev):
    K, N, I, H = 14336, 4096, 16384, 1024
    w, ws = (t[0] for t in pkg.synthetic_weights(1, N, K, dev, 5))
    w13, s13 = (t[0] for t in pkg.synthetic_weights(1, 2 * I, H, dev, 6))
    w2, s2 = (t[0] for t in pkg.synthetic_weights(1, H, I, dev, 7))
    rows = (2048, 1, 30, 33, 64, 100, 128, 129, 300, 700, 768, 1100)
    buf = [torch.empty(n, dtype=torch.uint8, device=dev) for n in (pkg.ops.mm_workspace_bytes(rows[0], K, N),
                                                                   pkg.ops.mlp_workspace_bytes(rows[0], H, I))]
    for M in rows:
        g = torch.Generator().manual_seed(M)
        x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
        assert torch.equal(pkg.mm_fp8(x, w, ws, workspace=buf[0]), pkg.mm_fp8(x, w, ws)), M
        x = torch.randn(M, H, generator=g).to(torch.bfloat16).to(dev)
        assert torch.equal(pkg.mlp_fp8(x, w13, s13, w2, s2, workspace=buf[1]), pkg.mlp_fp8(x, w13, s13, w2, s2)), M
