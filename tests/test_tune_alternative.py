"""Tuning entries of the pipelined kernel name the fastest kernel without scratch beside it: captured
calls, calls from a fifth stream and calls short of memory run that one."""
import pytest

PIPE, DIRECT = 64, 65


def _lines(path):
    return [l.split("\t") for l in open(path).read().splitlines() if not l.startswith("#")]


def test_entries_in_files(tmp_path):
    from ftd_amd import ftdx
    ctx = ftdx.CutlassComplexGemm()
    path = tmp_path / "tune.txt"
    ctx.tune_save(str(path))
    good = ["herk\t64\t32\t1\t0\t1\t64\t1\t1.5\t5\t0", "herk\t65\t32\t1\t0\t1\t64\t1\t1.5\t65\t1",
            "herk\t66\t32\t1\t0\t1\t64\t1\t1.5", "herk\t67\t32\t1\t0\t1\t65\t1\t1.5", "herk\t68\t32\t1\t0\t1\t4\t1\t1.5\t"]
    bad = ["herk\t64\t33\t1\t0\t1\t64\t1\t1.5\t5",           # one field of two
           "herk\t64\t33\t1\t0\t1\t64\t1\t1.5\t64\t1",       # needs scratch itself
           "herk\t64\t33\t1\t0\t1\t64\t1\t1.5\t9\t1",        # unknown
           "herk\t64\t33\t1\t0\t1\t64\t1\t1.5\t-1\t1",
           "herk\t64\t33\t1\t0\t1\t64\t1\t1.5\t5\t0\tmore",
           "herk\t64\t33\t1\t0\t1\t4\t1\t1.5\t5\t0",         # a tile has no use for one
           "herk\t64\t33\t1\t0\t1\t65\t1\t1.5\t5\t0"]
    with open(path, "a") as f:
        f.write("\n".join(good + bad) + "\n")
    assert ctx.tune_load(str(path)) == (len(good), len(bad))
    out = tmp_path / "again.txt"
    ctx.tune_save(str(out))
    assert sorted(_lines(out)) == sorted(l.rstrip("\t").split("\t") for l in good)


@pytest.mark.gpu
def test_tuning_keeps_an_alternative(dev, tmp_path):
    import torch
    from ftd_amd import ftdx
    N, K, B = 2048, 2048, 4
    ctx = ftdx.CutlassComplexGemm()
    A = torch.full((N * K * B,), 0x11, dtype=torch.uint8, device=dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    assert ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32, tune=True) == 0
    torch.cuda.synchronize()
    ctx.tune_save(str(tmp_path / "t.txt"))
    (line,) = _lines(tmp_path / "t.txt")
    assert len(line) == (11 if int(line[6]) == PIPE else 9), line
    assert int(line[6]) != PIPE or int(line[9]) in (0, 1, 2, 3, 4, 5, DIRECT)


@pytest.mark.gpu
@pytest.mark.parametrize("alt", ["", "\t0\t0", "\t1\t1", "\t2\t1", "\t3\t0", "\t5\t1", "\t65\t1"])
@pytest.mark.parametrize("K", [192, 200])
def test_captured_call_runs_the_alternative(oracle, dev, tmp_path, alt, K):
    import torch
    from ftd_amd import ftdx
    N, B = 300, 3
    path = tmp_path / "tune.txt"
    ctx = ftdx.CutlassComplexGemm()
    ctx.tune_save(str(path))
    with open(path, "a") as f:
        f.write(f"herk\t{N}\t{K}\t{B}\t0\t{1 if K % 16 == 0 else 4}\t{PIPE}\t1\t1.0{alt}\n")
    assert ctx.tune_load(str(path)) == (1, 0)
    qc = oracle.gen_qc_uniform(K, N * K * B)
    ref = torch.from_numpy(oracle.herk_f32(qc, N, K, B)).to(dev)
    A, C = torch.from_numpy(qc).to(dev), torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        for capture in (False, True):
            if capture:
                graph.capture_begin()
            assert ctx.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32, tune=False) == 0
            if capture:
                graph.capture_end()
                C.zero_()
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(C, ref)
            C.zero_()
