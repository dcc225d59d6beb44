"""Calls that a program captures into a HIP graph after one eager call of the same shape."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIPE = 64


def _replay(torch, graph, outs, refs, ctx):
    for _ in range(3):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for o, r in zip(outs, refs):
            assert torch.equal(o, r)


# rows that 16-byte loads cannot take, by their length and by their address
@pytest.mark.parametrize("K,shift", [(1000, 0), (1024, 1)])
@pytest.mark.parametrize("cached", [False, True])
def test_ragged_rows_after_an_eager_call(oracle, dev, tmp_path, K, shift, cached):
    """The eager call runs the pipelined kernel, which needs no padded rows; the captured one runs the
    fused tile on padded rows, in scratch that it cannot allocate."""
    import torch
    from ftd_amd import ftdx
    N, B = 1000, 12
    ctx = ftdx.CutlassComplexGemm()
    if cached:
        path = tmp_path / "tune.txt"
        ctx.tune_save(str(path))
        with open(path, "a") as f:
            f.write(f"herk\t{N}\t{K}\t{B}\t0\t4\t{PIPE}\t1\t1.0\n")
        assert ctx.tune_load(str(path)) == (1, 0)
    qc = oracle.gen_qc_uniform(K, N * K * B)
    buf = torch.zeros(qc.size + shift, dtype=torch.uint8, device=dev)
    A = buf[shift:]
    A.copy_(torch.from_numpy(qc))
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)

    def call():
        assert ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32, tune=False) == 0

    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        call()
        torch.cuda.synchronize()
        ref = C.clone()
        assert np.array_equal(ref[:1].cpu().numpy(), oracle.herk_f32(qc[:N * K], N, K, 1))
        with torch.cuda.graph(graph, stream=side):
            call()
        _replay(torch, graph, [C], [ref], ctx)


def test_ragged_gridding_after_an_eager_call(dev):
    import torch
    from ftd_amd import ftdx
    N, K, chan, pol, Ng, cell = 300, 1000, 3, 2, 512, 2e-3
    ctx = ftdx.CutlassComplexGemm()
    A = torch.randint(0, 256, (chan * pol * N * K,), dtype=torch.uint8, device=dev)
    uv = ((torch.rand((N * (N + 1) // 2, 2), device=dev) - 0.5) * Ng * cell * 0.2).contiguous()
    freq = torch.linspace(0.8e9, 1.3e9, chan, device=dev, dtype=torch.float64)
    grid = torch.zeros((chan, Ng, Ng, 2), device=dev)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        ftdx.herk_pol_grid(ctx, A, N, K, chan, pol, uv, freq, grid, Ng, cell)
        torch.cuda.synchronize()
        ref = grid.clone()
        assert float(ref.abs().max()) < 2 ** 24  # integer sums: any order of the atomics
        with torch.cuda.graph(graph, stream=side):
            ftdx.herk_pol_grid(ctx, A, N, K, chan, pol, uv, freq, grid, Ng, cell)
        _replay(torch, graph, [grid], [ref], ctx)


def test_streams_that_come_and_go(oracle, dev):
    """A context called from ever new streams: after the first four are idle their memory serves the
    next ones, and no more than four streams' rows are held."""
    import torch
    from ftd_amd import ftdx
    N, K, B = 2048, 2048, 2  # 12.6 MB of rows a stream
    qc = oracle.gen_qc_uniform(4, N * K * B)
    A = torch.from_numpy(qc).to(dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    ref = oracle.herk_f32(qc[:N * K], N, K, 1)
    ctx = ftdx.CutlassComplexGemm()
    streams = [torch.cuda.Stream() for _ in range(9)]
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    for s in streams:
        for _ in range(30):
            assert ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32, stream=s,
                            tune=False) == 0
        torch.cuda.synchronize()
        assert np.array_equal(C[:1].cpu().numpy(), ref)
        C.zero_()
        torch.cuda.synchronize()
    held = free0 - torch.cuda.mem_get_info()[0]
    assert held < 4 * 12.6e6 + 32e6, held


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("K", [2048, 2040])
def test_eager_calls_beside_a_capture(dev, grow, K):
    """A capture in progress (global mode) survives eager calls on another stream that need scratch for
    the first time, or more of it than before; K = 2040: rows that the fused tile would pad."""
    import torch
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()
    side, other, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    x = torch.arange(64.0, device=dev)
    y = torch.zeros_like(x)

    def call(N, K, B):
        A = torch.full((N * K * B,), 0x11, dtype=torch.uint8, device=dev)  # 1 + 1i
        C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
        torch.cuda.synchronize()
        return A, C, lambda: ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32,
                                      stream=other, tune=False)

    small, large = call(2048, K, 2), call(2048, K, 4)  # the pipelined kernel's
    if grow:
        assert small[2]() == 0
        torch.cuda.synchronize()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            y.copy_(x)
            assert large[2]() == 0
            y.add_(1.0)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, x + 1.0)
    assert bool((large[1][:, 0] == torch.tensor([2.0 * K, 0.0], device=dev)).all())
    assert bool((large[1][..., 0] == 2.0 * K).all())


def test_block_scaled_call_after_a_larger_one(dev):
    """A captured block-scaled call gets along with the scratch that an eager call of another, larger shape
    left: smaller chunks where its own would be more."""
    import torch
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()
    kw = dict(input=ftdx.InputPrecision.INT4, compute=ftdx.ComputePrecision.FP6, output="fp16")
    gen = torch.Generator(device=dev).manual_seed(2)

    def qc(n):
        return torch.randint(0, 256, (n,), generator=gen, dtype=torch.uint8, device=dev)

    N, K, B = 8192, 16384, 2  # one channel's fragments (210 MB) are a chunk
    big = torch.zeros((B, N * (N + 1) // 2, 2), dtype=torch.float16, device=dev)
    ftdx.herk_mx(ctx, qc(N * K * B), N, K, B, C=big, **kw)
    N, K, B = 1024, 1024, 200  # 328 MB in chunks of its own
    A = qc(N * K * B)
    C, ref = (torch.zeros((B, N * (N + 1) // 2, 2), dtype=torch.float16, device=dev) for _ in range(2))
    ftdx.herk_mx(ftdx.CutlassComplexGemm(), A, N, K, B, C=ref, **kw)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            ftdx.herk_mx(ctx, A, N, K, B, C=C, **kw)
        _replay(torch, graph, [C], [ref], ctx)


def test_padded_rows_of_a_captured_call_stay(oracle, dev):
    """A captured call on padded rows keeps its scratch: larger eager calls, which run the pipelined kernel,
    leave it where the replays read and write it."""
    import torch
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()

    def make(N, K, B):
        qc = oracle.gen_qc_uniform(K + B, N * K * B)
        A, C = torch.from_numpy(qc).to(dev), torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
        return C, lambda: ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32,
                                   tune=False), qc

    C, call, qc = make(1000, 1000, 12)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        assert call() == 0
        torch.cuda.synchronize()
        ref = C.clone()
        assert np.array_equal(ref[:1].cpu().numpy(), oracle.herk_f32(qc[:10 ** 6], 1000, 1000, 1))
        with torch.cuda.graph(graph, stream=side):
            assert call() == 0
        for K, B in ((1500, 20), (1999, 24)):
            D, big, _ = make(1000, K, B)
            assert big() == 0
            junk = [torch.full((1 << 22,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(16)]
            _replay(torch, graph, [C], [ref], ctx)
            assert all(bool((j == 0x5A).all()) for j in junk)
