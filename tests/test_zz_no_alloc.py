"""llmr_batch_matmul_noalloc, the GEMM entry point that allocates nothing:
its scratch is the library's fixed device array. Each case calls it twice in
a row through the C-ABI, the second time with a smaller input, and compares
every output with llmr_batch_matmul's on the same inputs: bit for bit where
both run the same kernels or the no-allocation call runs the one-pass
kernels in place of the two-pass path (the same bits), to f32 summation
order where it runs fewer K splits. A fresh context's no-allocation calls
leave the device's free memory unchanged, and calls of one context on two
streams are ordered around the shared scratch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

F32, F16, BF16 = 0, 1, 30


def _weights(dev, wtype, rows, K, seed):
    from llmr_amd import glue, gguf, synth
    if wtype == 12:
        return glue.synth_q4k(rows, K, seed, device=dev)
    return torch.from_numpy(gguf.quantize(synth.normal(seed, 2, rows * K, 0.02), wtype)).to(dev)


def _x(dev, M, K, xtype, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    return (x if xtype == F32 else x.to(torch.float16 if xtype == F16 else torch.bfloat16)).to(dev)


def _both(dev, w, wtype, x, xtype, N, row_offset=0):
    from llmr_amd import ops
    g = ops.default_graph()
    g.bind_stream()
    M, K = x.shape
    y_ref = torch.full((M, N), 7.0, dtype=torch.float32, device=dev)
    y = torch.full((M, N), -7.0, dtype=torch.float32, device=dev)
    g.ctx.batch_matmul(w.data_ptr(), wtype, x.data_ptr(), xtype, y_ref.data_ptr(), N, K, M, row_offset)
    g.ctx.batch_matmul_noalloc(w.data_ptr(), wtype, x.data_ptr(), xtype, y.data_ptr(), N, K, M, row_offset)
    torch.cuda.synchronize()
    return y, y_ref


# (wtype, xtype, N, K, (M first call, M second call), row_offset, what the
# scratch holds). Where llmr_batch_matmul's plan fits the array both calls run
# the same kernels (same bits); a launch whose weight image does not fit runs
# the one-pass kernels (same bits as the two-pass path); one whose split-K
# partials or partial tiles do not fit runs fewer splits or another kernel (the
# same sums in another order: compared to f32 rounding, far inside the GEMM bar
# of relative L2 1e-2; `exact` False for that launch). tests/c/plan_check.cpp
# pins what each of these launches holds in the scratch.
CASES = [
    (8, F32, 3072, 3072, (256, 64), 0, (True, True), "nothing (the few-token kernel)"),
    (12, F32, 3840, 10240, (64, 33), 0, (True, True), "packed activations and split-K partials"),
    (12, F32, 4096, 1024, (4096, 2304), 8, (True, True), "f32 activations as bf16 + the weight image"),
    (12, BF16, 12288, 3072, (2560, 2304), 0, (True, True), "nothing: one-pass in place of a 75 MB weight image"),
    (12, BF16, 3072, 3072, (4608, 2048), 0, (True, False), "the weight image; then no partials"),
    (8, F16, 1000, 14400, (200, 40), 4, (True, True), "split-K partials, ragged N"),
    (8, BF16, 3840, 5120, (600, 513), 0, (False, False), "partial tiles, in fewer parts"),
]


@pytest.mark.parametrize("wtype,xtype,N,K,Ms,row_offset,exact,what", CASES)
def test_noalloc_matches_batch_matmul_twice(dev, wtype, xtype, N, K, Ms, row_offset, exact, what):
    from conftest import rel_l2
    w = _weights(dev, wtype, N + row_offset, K, 60 + wtype)
    for i, M in enumerate(Ms):
        x = _x(dev, M, K, xtype, 1000 * i + M)
        print(f"noalloc wtype={wtype} xtype={xtype} M={M} N={N} K={K} ({what})", flush=True)
        y, y_ref = _both(dev, w, wtype, x, xtype, N, row_offset)
        assert bool(torch.isfinite(y_ref).all())
        assert bool(torch.isfinite(y).all())
        err = rel_l2(y.cpu().numpy(), y_ref.cpu().numpy())
        same = torch.equal(y, y_ref)
        print(f"  rel L2 {err:.2e}, identical {same}")
        assert err <= 1e-5, (M, err)
        assert same or not exact[i], M


def test_noalloc_f32_beyond_scratch_runs_tiled(dev):
    """f32 activations of 4608 x 4096 would need a 36 MiB 16-bit copy for the
    persistent kernels, more than the 32 MiB array: the call runs the tiled
    kernel, which rounds them in registers to the same operands, so it agrees
    with llmr_batch_matmul to f32 summation order."""
    from conftest import rel_l2
    N, K, M = 4096, 4096, 4608
    w = _weights(dev, 12, N, K, 77)
    x = _x(dev, M, K, F32, 5)
    print("noalloc f32 4608 x 4096 x 4096 Q4_K (tiled in place of the persistent kernels)", flush=True)
    y, y_ref = _both(dev, w, 12, x, F32, N)
    assert bool(torch.isfinite(y).all())
    err = rel_l2(y.cpu().numpy(), y_ref.cpu().numpy())
    print(f"  rel L2 {err:.2e}")
    assert err <= 1e-5


def test_noalloc_allocates_nothing_on_a_fresh_context(dev):
    """A context that has never run a GEMM calls only llmr_batch_matmul_noalloc,
    on launches whose plans use scratch (split-K partials, a 16-bit copy of f32
    activations, a weight image, partial tiles): the device's free memory is the same before
    and after. (The kernels' code is loaded first through another context.)"""
    from llmr_amd import capi, ops
    cases = [(12, F32, 512, 10240, 64), (12, F32, 4096, 1024, 2304), (12, BF16, 3072, 3072, 4608),
             (8, BF16, 3840, 5120, 600)]
    data = []
    for wtype, xtype, N, K, M in cases:
        w = _weights(dev, wtype, N, K, 90 + wtype)
        x = _x(dev, M, K, xtype, 3 + M)
        y = torch.empty((M, N), dtype=torch.float32, device=dev)
        data.append((w, wtype, x, xtype, y, N, K, M))
    warm = ops.default_graph()
    warm.bind_stream()
    for w, wtype, x, xtype, y, N, K, M in data:  # load every kernel's code
        warm.ctx.batch_matmul_noalloc(w.data_ptr(), wtype, x.data_ptr(), xtype, y.data_ptr(), N, K, M, 0)
    torch.cuda.synchronize()
    ctx = capi.Context(0)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    free0 = torch.cuda.mem_get_info()[0]
    for w, wtype, x, xtype, y, N, K, M in data:
        print(f"fresh context noalloc wtype={wtype} xtype={xtype} M={M} N={N} K={K}", flush=True)
        ctx.batch_matmul_noalloc(w.data_ptr(), wtype, x.data_ptr(), xtype, y.data_ptr(), N, K, M, 0)
    torch.cuda.synchronize()
    free1 = torch.cuda.mem_get_info()[0]
    ctx.close()
    assert free1 == free0, (free0, free1)
    assert all(bool(torch.isfinite(d[4]).all()) for d in data)


def test_noalloc_two_streams_of_one_context(dev):
    """Two no-allocation calls whose plans use the scratch (split-K partials),
    issued on two streams of one context one after the other: the second
    waits for the first stream's work up to the switch, so both results are
    llmr_batch_matmul's."""
    from llmr_amd import capi
    N, K = 3840, 10240
    w = _weights(dev, 12, N, K, 31)
    xs = [_x(dev, 64, K, F32, 11), _x(dev, 64, K, F32, 12)]
    ys = [torch.full((64, N), -1.0, device=dev) for _ in xs]
    refs = [torch.empty((64, N), device=dev) for _ in xs]
    ctx = capi.Context(0)
    s0, s1 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    print("noalloc on two streams of one context: 64 x 3840 x 10240 Q4_K f32 (split-K partials)", flush=True)
    for st, x, y in ((s0, xs[0], ys[0]), (s1, xs[1], ys[1])):
        ctx.set_stream(st.cuda_stream)
        ctx.batch_matmul_noalloc(w.data_ptr(), 12, x.data_ptr(), F32, y.data_ptr(), N, K, 64, 0)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for x, r in zip(xs, refs):
        ctx.batch_matmul(w.data_ptr(), 12, x.data_ptr(), F32, r.data_ptr(), N, K, 64, 0)
    torch.cuda.synchronize()
    ctx.close()
    for y, r in zip(ys, refs):
        assert torch.equal(y, r)


def test_captured_gemm_takes_no_workspace(dev):
    """Launches whose tiles are cut along K outside a capture (partial tiles in
    the workspace) need none under one: a context that holds no workspace
    captures llmr_batch_matmul, and llmr_batch_matmul_noalloc after the scratch
    was used on another stream; every replay, with the context's own work and a
    larger workspace between, gives the eager result to f32 summation order."""
    from conftest import rel_l2
    from llmr_amd import capi, ops
    wtype, N, K, M = 8, 3840, 5120, 600  # 45 tiles, cut into fewer parts within the scratch
    w, x = _weights(dev, wtype, N, K, 41), _x(dev, M, K, BF16, 42)
    ws, xs = _weights(dev, 12, 512, 10240, 43), _x(dev, 64, 10240, F32, 44)  # split-K partials
    g = ops.default_graph()
    g.bind_stream()
    y_ref = torch.empty((M, N), device=dev)
    g.ctx.batch_matmul(w.data_ptr(), wtype, x.data_ptr(), BF16, y_ref.data_ptr(), N, K, M, 0)
    ys = torch.empty((64, 512), device=dev)
    ctx = capi.Context(0)
    side = torch.cuda.Stream()
    main = torch.cuda.current_stream().cuda_stream

    def scratch_call():
        ctx.batch_matmul_noalloc(ws.data_ptr(), 12, xs.data_ptr(), F32, ys.data_ptr(), 512, 10240, 64, 0)

    ctx.set_stream(main)
    scratch_call()
    torch.cuda.synchronize()
    ctx.set_stream(side.cuda_stream)
    y, y_na = (torch.empty((M, N), device=dev) for _ in range(2))
    graph = torch.cuda.CUDAGraph()
    print("capture of 600 x 3840 x 5120 Q8_0 bf16", flush=True)
    with torch.cuda.graph(graph, stream=side):
        ctx.batch_matmul(w.data_ptr(), wtype, x.data_ptr(), BF16, y.data_ptr(), N, K, M, 0)
        ctx.batch_matmul_noalloc(w.data_ptr(), wtype, x.data_ptr(), BF16, y_na.data_ptr(), N, K, M, 0)
    ctx.set_stream(main)
    y_big = torch.empty((2 * M, N), device=dev)
    for i in range(3):
        y.fill_(7.0)
        y_na.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        for t in (y, y_na):
            assert rel_l2(t.cpu().numpy(), y_ref.cpu().numpy()) <= 1e-5, i
        scratch_call()
        ctx.batch_matmul(w.data_ptr(), wtype, x.data_ptr(), BF16, y_big[i * 4:].data_ptr(), N, K, M - 100 * (2 - i), 0)
        torch.cuda.synchronize()
    ctx.close()
