"""INT4 HERK without a forced tile: the pipelined kernel over E3M2 fragment rows and the direct
kernel for small problems, bit-exact against the CPU oracle.  A tuning cache entry names the
kernel, so every size runs on the one under test whatever the library would choose."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIPE, DIRECT = 64, 65


def _bits(x):
    return x.view(np.uint32 if x.dtype == np.float32 else np.uint16)


def _context(tmp_path, shapes, kernel):
    """A context whose tuning cache sends each (N, K, batch) to `kernel`, for both output types
    and for rows with and without 16-byte loads."""
    from ftd_amd import ftdx
    path = tmp_path / "tune.txt"
    ctx = ftdx.CutlassComplexGemm()
    ctx.tune_save(str(path))
    with open(path, "a") as f:
        for N, K, B in shapes:
            for fp16 in (0, 1):
                for rows in (1, 4):
                    f.write(f"herk\t{N}\t{K}\t{B}\t{fp16}\t{rows}\t{kernel}\t1\t1.0\n")
    assert ctx.tune_load(str(path)) == (4 * len(shapes), 0)
    return ctx


def _run(ctx, A, C, N, K, B, **kw):
    from ftd_amd import ftdx
    import torch
    out = ftdx.OutputPrecision.FP32 if C.dtype == torch.float32 else ftdx.OutputPrecision.FP16
    assert ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=out, tune=False, **kw) == 0


# tile (128 / 32 rows), group (32), stage (64) and segment (16) edges; K past the sample counts
# where the stores turn non-temporal (320 and 448) and where the direct kernel takes 16 waves (961)
SHAPES = [(1, 16, 3), (31, 17, 2), (33, 63, 2), (65, 64, 2), (127, 65, 1), (128, 128, 2), (129, 200, 2),
          (193, 321, 1), (257, 449, 1), (300, 1000, 1), (520, 130, 1), (640, 64, 1)]


@pytest.mark.parametrize("kernel", [PIPE, DIRECT])
@pytest.mark.parametrize("N,K,B", SHAPES)
def test_kernel_edges_bit_exact(oracle, dev, tmp_path, kernel, N, K, B):
    import torch
    ctx = _context(tmp_path, [(N, K, B)], kernel)
    qc = oracle.gen_bytes(N * 3 + K, N * K * B)  # every byte, -0 nibbles among them
    ref = oracle.herk_f32(qc, N, K, B)
    # rows at a 16-byte boundary, and one byte past it
    for shift in (0, 1):
        buf = torch.zeros(shift + qc.size, dtype=torch.uint8, device=dev)
        A = buf[shift:]
        A.copy_(torch.from_numpy(qc))
        C = torch.full((B, N * (N + 1) // 2, 2), 7.0, device=dev)
        _run(ctx, A, C, N, K, B)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(C.cpu().numpy()), _bits(ref)), shift
    H = torch.full((B, N * (N + 1) // 2, 2), 7.0, device=dev, dtype=torch.float16)
    _run(ctx, A, H, N, K, B, alpha=2.0 ** -10)
    torch.cuda.synchronize()
    want = (ref.astype(np.float64) * 2.0 ** -10).astype(np.float16)
    assert np.array_equal(H.cpu().numpy(), want)


@pytest.mark.parametrize("kernel", [PIPE, DIRECT])
def test_alpha_beta(oracle, dev, tmp_path, kernel):
    """alpha first, then one fma with beta; powers of two keep every step exact."""
    import torch
    N, K, B = 200, 96, 2
    ctx = _context(tmp_path, [(N, K, B)], kernel)
    qc = oracle.gen_qc_uniform(4, N * K * B)
    ref = oracle.herk_f32(qc, N, K, B).astype(np.float64)
    A = torch.from_numpy(qc).to(dev)
    C = torch.full((B, N * (N + 1) // 2, 2), 3.0, device=dev)
    _run(ctx, A, C, N, K, B, alpha=0.5, beta=-2.0)
    torch.cuda.synchronize()
    assert np.array_equal(C.cpu().numpy(), (0.5 * ref - 6.0).astype(np.float32))


@pytest.mark.parametrize("kernel", [PIPE, DIRECT])
def test_long_coherent_sums_stay_exact(dev, tmp_path, kernel):
    """Sums of one sign up to 98 x 160016 = 15.7e6, close below 2^24, odd ones among them: the
    matrix cores' internal sum must not drop a low bit next to a large accumulator."""
    import torch
    N, K, B = 40, 160016, 1
    ctx = _context(tmp_path, [(N, K, B)], kernel)
    gen = torch.Generator(device="cpu").manual_seed(3)
    v = torch.randint(6, 8, (2, N, K), generator=gen, dtype=torch.int32)
    v[:, 0] = 7
    v[:, 1, 1:] = 7
    A = ((v[0] << 4) | v[1]).to(torch.uint8).to(dev)
    C = torch.empty((B, N * (N + 1) // 2, 2), device=dev)
    _run(ctx, A, C, N, K, B)
    torch.cuda.synchronize()
    re, im = v.to(torch.float64)
    i, j = torch.from_numpy(np.stack(np.tril_indices(N)))
    want = torch.stack([(re @ re.T + im @ im.T)[i, j], (im @ re.T - re @ im.T)[i, j]], -1)
    want[i == j, 1] = 0.0
    assert float(want.max()) == 98.0 * K < 2 ** 24
    assert torch.equal(C[0].cpu().double(), want)


def test_pipe_batches_in_chunks(dev, tmp_path):
    """More channels than one 160 MB chunk of fragment rows: every channel is converted and
    multiplied, checked by weighted checksums and exact rows."""
    import torch
    from ftd_amd import selfcheck
    N, K, B = 1000, 2000, 60  # 3.1 MB of rows per channel, 51 channels per chunk at most
    ctx = _context(tmp_path, [(N, K, B)], PIPE)
    A = selfcheck.qc_uniform(N * K * B, 11, dev)
    C = torch.empty((B, N * (N + 1) // 2, 2), device=dev)
    _run(ctx, A, C, N, K, B)
    torch.cuda.synchronize()
    res = selfcheck.check_herk(torch, A, C, N, K, B, rows=[0, 127, 128, 999], row_channels=[0, 50, 51, 59])
    assert res["ok"], res


def test_streams_do_not_share_fragment_rows(oracle, dev, tmp_path):
    """One context on six streams without waiting in between: each has rows of its own or takes
    the fused tile, so no call overwrites another's."""
    import torch
    N, K, B = 700, 256, 4
    ctx = _context(tmp_path, [(N, K, B)], PIPE)
    data = [oracle.gen_qc_uniform(20 + s, N * K * B) for s in range(6)]
    A = [torch.from_numpy(q).to(dev) for q in data]
    C = [torch.zeros((B, N * (N + 1) // 2, 2), device=dev) for _ in data]
    streams = [torch.cuda.Stream() for _ in data]
    torch.cuda.synchronize()
    for _ in range(5):
        for s, a, c in zip(streams, A, C):
            _run(ctx, a, c, N, K, B, stream=s)
    torch.cuda.synchronize()
    for q, c in zip(data, C):
        assert np.array_equal(_bits(c.cpu().numpy()), _bits(oracle.herk_f32(q, N, K, B)))


@pytest.mark.parametrize("kernel", [None, PIPE])
def test_captured_call_keeps_no_scratch(oracle, dev, tmp_path, kernel):
    """A call captured by the program runs without the context's fragment rows: replays stay right
    after a larger call replaced them, and after the context gave them back."""
    import torch
    from ftd_amd import ftdx
    N, K, B = 512, 512, 6
    ctx = _context(tmp_path, [(N, K, B)] if kernel else [], kernel)
    qc = oracle.gen_qc_uniform(9, N * K * B)
    ref = oracle.herk_f32(qc, N, K, B)
    A = torch.from_numpy(qc).to(dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        _run(ctx, A, C, N, K, B)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            _run(ctx, A, C, N, K, B)
        big = torch.zeros(2048 * 512 * 16, dtype=torch.uint8, device=dev)
        D = torch.empty((16, 2048 * 2049 // 2, 2), device=dev)
        for done in (lambda: _run(ctx, big, D, 2048, 512, 16), ctx.end_herk, ctx.end_herk):
            C.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(_bits(C.cpu().numpy()), _bits(ref))
            done()
            torch.cuda.synchronize()
    assert ctx.query_config(N, K, B)[0] == (kernel or ftdx.TILE_128x128_K64)


def test_kernel_ids_are_not_settings():
    """The two kernels are the library's choice or the autotuner's, not a tile a caller can force."""
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()
    for k in (PIPE, DIRECT):
        with pytest.raises(ftdx.FtdxError):
            ctx.set_launch_config(k, 1)


def test_choice_by_size_bit_exact(oracle, dev):
    """The library's own choice over sizes on each side of its lines: the direct kernel, the fused
    tile and the pipelined kernel all give the oracle's bytes."""
    import torch
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()
    for N, K, B in [(64, 64, 1), (128, 1024, 16), (256, 4000, 3), (512, 1024, 20), (512, 1000, 20), (700, 2048, 1),
                    (1001, 333, 3), (96, 8, 2), (40, 0, 2)]:
        qc = oracle.gen_qc_uniform(N + K, N * K * B)
        A = torch.from_numpy(qc).to(dev) if K else torch.zeros(1, dtype=torch.uint8, device=dev)
        C = torch.full((B, N * (N + 1) // 2, 2), 5.0, device=dev)
        _run(ctx, A, C, N, K, B)
        torch.cuda.synchronize()
        ref = oracle.herk_f32(qc, N, K, B) if K else np.zeros(C.shape, np.float32)
        assert np.array_equal(_bits(C.cpu().numpy()), _bits(ref)), (N, K, B)


# A plan of large problems runs the pipelined kernel; the small ones among them take its edges
# (no samples, rows shorter than one 16-byte segment, tile and stage remainders, unaligned rows).
GROUP_EDGES = [(1, 5), (40, 0), (33, 15), (64, 16), (65, 17), (127, 65), (129, 64), (257, 449), (31, 1000)]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("fp16", [False, True])
def test_grouped_fragment_rows_bit_exact(oracle, dev, graph, fp16):
    import torch
    from ftd_amd import ftdx
    out = ftdx.OutputPrecision.FP16 if fp16 else ftdx.OutputPrecision.FP32
    dt = torch.float16 if fp16 else torch.float32
    ctx, probs, refs = ftdx.CutlassComplexGemm(), [], []
    for i, (N, K) in enumerate(GROUP_EDGES):
        qc = oracle.gen_bytes(70 + i, max(N * K, 1))
        buf = torch.zeros(qc.size + i, dtype=torch.uint8, device=dev)
        buf[i:].copy_(torch.from_numpy(qc))
        C = torch.full((N * (N + 1) // 2, 2), float("nan"), dtype=dt, device=dev)
        probs.append((buf[i:], C, N, K, 0.5 if i % 2 else 1.0, 0.0))
        alpha = probs[-1][4]
        ref = (oracle.herk_f16 if fp16 else oracle.herk_f32)(qc[:N * K], N, K, 1, alpha=alpha) if K else None
        refs.append(None if ref is None else ref[0])
    big = [(2048, 2048)] * 24
    Ab = torch.randint(0, 256, (2048 * 2048,), dtype=torch.uint8, device=dev)
    Cb = [torch.empty((2048 * 2049 // 2, 2), dtype=dt, device=dev) for _ in big]
    probs += [(Ab, C, N, K, 1.0, 0.0) for C, (N, K) in zip(Cb, big)]
    plan = ftdx.GroupedPlan(ctx, probs, output=out, use_graph=graph)
    assert plan.info()["workgroups"] > 24 * 136  # a workgroup per tile: not the persistent kernel
    fused = torch.empty_like(Cb[0])
    one = ftdx.GroupedPlan(ctx, [(Ab, fused, 2048, 2048, 1.0, 0.0)], output=out, tile_config=0, use_graph=False)
    one.run()
    for _ in range(3):
        for p in probs:
            p[1].fill_(float("nan"))
        plan.run()
        torch.cuda.synchronize()
        for p, ref in zip(probs, refs):
            got = p[1].cpu().numpy()
            assert np.array_equal(_bits(got), _bits(np.zeros_like(got) if ref is None else ref)), (p[2], p[3])
        for C in Cb:
            assert torch.equal(C, fused)
