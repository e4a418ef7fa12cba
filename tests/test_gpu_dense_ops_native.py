"""The dense ops' native path against the general one: the same bits for every form both accept, and packed copies that
follow their weights."""
import gc

import pytest
import torch
from torch.multiprocessing.reductions import StorageWeakRef

pytestmark = pytest.mark.gpu


def weights(dev, n, k, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(n, k, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(dev)
    return w, ((torch.rand(-(-n // 128), -(-k // 128), generator=g) + 0.5) * 0.01).to(dtype).to(dev)


@pytest.mark.parametrize("M,K,N", [(1, 128, 16), (32, 7168, 1536), (5, 256, 1040), (130, 384, 272)])
@pytest.mark.parametrize("form", ["plain", "fp32 scales", "strided weight", "strided input", "strided output", "float64 scales"])
def test_mm_forms(pkg, dev, M, K, N, form):
    w, s = weights(dev, N, K, M + K, {"fp32 scales": torch.float32, "float64 scales": torch.float64}.get(form, torch.bfloat16))
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(N)).to(torch.bfloat16).to(dev)
    if form == "strided weight":
        w = w.t().contiguous().t()
    if form == "strided input":
        x = torch.cat([x, x], 1)[:, :K]
    a, b = torch.zeros(2, M, 2 * N, dtype=torch.bfloat16, device=dev)
    a, b = (t[:, :N] if form == "strided output" else t[:, :N].contiguous() for t in (a, b))
    r = torch.ops.my_ops.mm_w8a16_dq_forward(x, w, s, a, 128)
    assert r.data_ptr() == a.data_ptr()
    torch.ops.my_ops._mm_general(x, w, s, b, 128)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and a.abs().max() > 0


@pytest.mark.parametrize("M,H,I", [(1, 128, 128), (3, 256, 384), (140, 384, 512)])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_mlp_forms(pkg, dev, M, H, I, scale_dtype):
    (g, gs), (u, us), (d, ds) = (weights(dev, I, H, i, scale_dtype) for i in range(3))
    x = torch.randn(M, H, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(dev)
    a, b = torch.zeros(2, M, H, dtype=torch.bfloat16, device=dev)
    torch.ops.my_ops.mlp_w8a16_dq_forward(x, g, u, d, gs, us, ds, a, 128)
    torch.ops.my_ops._mlp_general(x, g, u, d, gs, us, ds, b, 128)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and a.abs().max() > 0


def test_packed_copy_follows_its_weight(pkg, dev):
    x = torch.randn(4, 256, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    w, s = weights(dev, 128, 256, 2)
    run = lambda: torch.ops.my_ops.mm_w8a16_dq_forward(x, w, s, torch.empty(4, 128, dtype=torch.bfloat16, device=dev), 128)
    first = run()
    s.mul_(2)                                             # an in-place write moves the version counter
    assert torch.equal(run(), first * 2)
    w.copy_(torch.zeros_like(w))
    assert run().abs().max() == 0
    del w
    w, s = weights(dev, 128, 256, 3)                      # new storages, possibly on the old addresses
    out = torch.empty(4, 128, dtype=torch.bfloat16, device=dev)
    torch.ops.my_ops._mm_general(x, w, s, out, 128)
    assert torch.equal(run(), out)


def test_what_was_refused_stays_refused(pkg, dev):
    x = torch.zeros(4, 256, dtype=torch.bfloat16, device=dev)
    w, s = weights(dev, 128, 256, 2)
    out = torch.empty(4, 128, dtype=torch.bfloat16, device=dev)
    for bad in [(x.float(), w, s, out, 128), (x, w.to(torch.bfloat16), s, out, 128), (x, w, s, out.float(), 128), (x, w, s, out, 0)]:
        with pytest.raises((RuntimeError, TypeError, ValueError)):
            torch.ops.my_ops.mm_w8a16_dq_forward(*bad)


def flat_views(dev, *parts):
    """The parts as views of one storage, each 512-byte aligned."""
    sizes = [(p.numel() * p.element_size() + 511) // 512 * 512 for p in parts]
    flat = torch.zeros(sum(sizes), dtype=torch.uint8, device=dev)
    views, at = [], 0
    for p, n in zip(parts, sizes):
        v = flat[at:at + p.numel() * p.element_size()].view(p.dtype).view(p.shape)
        v.copy_(p)
        views.append(v)
        at += n
    return views


@pytest.mark.parametrize("form", ["one flat buffer", "parameters"])
@pytest.mark.parametrize("op", ["mm", "mlp", "experts"])
def test_packed_copy_does_not_keep_its_sources_alive(pkg, dev, op, form):
    E, I, H = 4, 128, 256
    x = torch.randn(3, H, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    lead = (E,) if op == "experts" else ()
    tensors = []
    for i in range(1 if op == "mm" else 3):
        w, s = weights(dev, I * max(1, *lead, 1), H, i, torch.float32)
        tensors += [w.view(*lead, I, H), s.view(*lead, I // 128, H // 128)]
    if form == "parameters":
        tensors = [torch.nn.Parameter(t, requires_grad=t.dtype == torch.float32) for t in tensors]
    else:
        tensors = flat_views(dev, *tensors)
    alive = [StorageWeakRef(t.untyped_storage()) for t in tensors]
    my_ops = torch.ops.my_ops
    ids = torch.zeros(3, 1, dtype=torch.int32, device=dev)
    if op == "mm":
        my_ops.mm_w8a16_dq_forward(x, *tensors, torch.empty(3, I, dtype=torch.bfloat16, device=dev), 128)
    elif op == "mlp":
        my_ops.mlp_w8a16_dq_forward(x, *tensors[::2], *tensors[1::2], torch.empty_like(x), 128)
    else:
        my_ops.fused_moe_fused_experts(torch.empty_like(x), x, None, None, *tensors[::2], *tensors[1::2], ids, ids.float(), None,
                                       None, None, 128, E, 1, False, 1, 1, None, None, None, False)
    torch.cuda.synchronize()
    del tensors, w, s
    gc.collect()
    assert all(a.expired() for a in alive)


@pytest.mark.parametrize("op", ["mm", "mlp", "experts"])
def test_updates_of_a_live_weight_leave_one_packed_copy(pkg, dev, op):
    E, I, H = 4, 512, 1024
    lead = (E,) if op == "experts" else ()
    my_ops = torch.ops.my_ops
    x = torch.randn(5, H, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    ids = torch.randint(0, E, (5, 1), generator=torch.Generator().manual_seed(2), dtype=torch.int32).to(dev)
    tensors = []
    for i in range(1 if op == "mm" else 3):
        w, s = weights(dev, I * max(1, *lead, 1), H, i)
        tensors += [w.view(*lead, I, H), s.view(*lead, I // 128, H // 128)]
    fresh = [[weights(dev, t.numel() // H, H, 10 * k + i)[0].view(t.shape) for i, t in enumerate(tensors[::2])] for k in range(6)]

    def run(ts):
        out = torch.empty(5, I if op == "mm" else H, dtype=torch.bfloat16, device=dev)
        if op == "mm":
            return my_ops.mm_w8a16_dq_forward(x, *ts, out, 128)
        if op == "mlp":
            return my_ops.mlp_w8a16_dq_forward(x, *ts[::2], *ts[1::2], out, 128)
        return my_ops.fused_moe_fused_experts(out, x, None, None, *ts[::2], *ts[1::2], ids, ids.float() + 1, None, None, None,
                                              128, E, 1, False, 1, 1, None, None, None, False)

    run(tensors)
    gc.collect()
    before = torch.cuda.memory_allocated()
    for new in fresh:                                     # a weight sync: the same tensors, written again
        for t, n in zip(tensors[::2], new):
            t.copy_(n)
        tensors[1].mul_(0.5)
        got = run(tensors)
        clones = [t.clone() for t in tensors]
        assert torch.equal(got, run(clones))
        del got, clones
        run(tensors)                                      # (a call drops the entries of freed tensors)
    gc.collect()
    assert torch.cuda.memory_allocated() <= before + 4096


def one_mm(dev, seed, M=8, K=1024, N=512):
    w, s = weights(dev, N, K, seed)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(dev)
    return x, w, s, torch.empty(M, N, dtype=torch.bfloat16, device=dev)


@pytest.mark.parametrize("block", [128, 256])            # the C++ table, the Python one
def test_a_call_on_another_stream_waits_for_the_packing(pkg, dev, block):
    my_ops = torch.ops.my_ops
    x, w, s, out = one_mm(dev, 1, K=4096, N=4096)
    want = my_ops.mm_w8a16_dq_forward(x, w.clone(), s.clone(), torch.empty_like(out), block)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(20_000_000)                     # the packing lies behind some milliseconds of other work
        first = my_ops.mm_w8a16_dq_forward(x, w, s, torch.empty_like(out), block)
    with torch.cuda.stream(b):
        second = my_ops.mm_w8a16_dq_forward(x, w, s, torch.empty_like(out), block)
    w.record_stream(a)
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)
    # an update made and packed on one stream is seen by a call on the other
    with torch.cuda.stream(b):
        torch.cuda._sleep(20_000_000)
        s.mul_(2)
        my_ops.mm_w8a16_dq_forward(x, w, s, out, block)
        done = torch.cuda.Event()
        done.record()
    with torch.cuda.stream(a):
        a.wait_event(done)
        second = my_ops.mm_w8a16_dq_forward(x, w, s, torch.empty_like(out), block)
    torch.cuda.synchronize()
    assert torch.equal(out, want * 2) and torch.equal(second, want * 2)


@pytest.mark.parametrize("block", [128, 256])
def test_captured_calls_with_packed_known_and_new_weights(pkg, dev, block):
    """A weight packed before the capture is used as it is, one that is new to the capture is packed inside the graph and
    left alone by eager calls, and an eager refill after an update reaches the graph's copy."""
    my_ops = torch.ops.my_ops
    known, new = one_mm(dev, 3), one_mm(dev, 4)
    run = lambda t, out=None: my_ops.mm_w8a16_dq_forward(*t[:3], t[3] if out is None else out, block)
    want = [run((t[0], t[1].clone(), t[2].clone(), torch.empty_like(t[3]))) for t in (known, new)]
    run(known)
    torch.cuda.synchronize()
    held = my_ops._packed_weight_bytes()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(known)
        run(new)
    assert my_ops._packed_weight_bytes() <= held          # (less, if the clones' entries went)
    eager = run(new, torch.empty_like(new[3]))            # before the graph has run at all
    torch.cuda.synchronize()
    assert torch.equal(eager, want[1])
    for _ in range(3):
        known[3].zero_()
        new[3].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(known[3], want[0]) and torch.equal(new[3], want[1])
        assert torch.equal(run(known, torch.empty_like(known[3])), want[0])
    if block != 128:                                      # (the Python table replaces the copy of an updated weight)
        return
    for t in (known, new):
        t[2].mul_(2)
        run(t, torch.empty_like(t[3]))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(known[3], want[0] * 2) and torch.equal(new[3], want[1] * 2)


def test_capture_begun_while_the_packing_still_runs(pkg, dev):
    my_ops = torch.ops.my_ops
    x, w, s, out = one_mm(dev, 5)
    want = my_ops.mm_w8a16_dq_forward(x, w.clone(), s.clone(), torch.empty_like(out), 128)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)
    my_ops.mm_w8a16_dq_forward(x, w, s, torch.empty_like(out), 128)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        graph.capture_begin()
        my_ops.mm_w8a16_dq_forward(x, w, s, out, 128)
        graph.capture_end()
    out.zero_()
    torch.cuda.synchronize()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        out.zero_()


@pytest.mark.parametrize("op", ["mm", "mlp"])
def test_a_weight_is_packed_once_whatever_form_its_calls_take(pkg, dev, op):
    my_ops = torch.ops.my_ops
    I, H, M = 256, 512, 6
    ts = []
    for i in range(1 if op == "mm" else 3):
        ts += weights(dev, I, H, i)
    x = torch.randn(M, H, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    fn = my_ops.mm_w8a16_dq_forward if op == "mm" else my_ops.mlp_w8a16_dq_forward
    args = tuple(ts) if op == "mm" else (*ts[::2], *ts[1::2])
    width = I if op == "mm" else H
    call = lambda f, x: f(x, *args, torch.empty(M, 2 * width, dtype=torch.bfloat16, device=dev)[:, :width], 128)
    pkg.invalidate_weight_cache()
    want = fn(x, *args, torch.empty(M, width, dtype=torch.bfloat16, device=dev), 128).clone()
    held = my_ops._packed_weight_bytes()
    assert held == sum(t.nbytes for t in ts[::2]) + 4 * sum(t.numel() for t in ts[1::2])
    assert torch.equal(call(fn, x), want)                                         # strided output
    assert torch.equal(call(fn, torch.cat([x, x], 1)[:, :H]), want)               # strided input
    if op == "mlp":
        assert torch.equal(call(my_ops.mlp_w8a8_quant_forward, x), want)
    pkg.set_expert_numerics("w8a16")
    try:
        other = call(fn, x)
    finally:
        pkg.set_expert_numerics("w8a8")
    assert (other.float() - want.float()).norm() < 0.1 * want.float().norm()
    assert my_ops._packed_weight_bytes() == held and len(pkg._my_ops._weights) == 0
