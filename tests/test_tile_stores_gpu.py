"""Which stores a HERK tile's interior takes (staged through LDS, plain or non-temporal from the
accumulators) follows from the samples of all K segments, the output's size and the number of
tiles: the same bits on each side of those lines."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pol_sum(ctx, A, N, K, ch, pol, out, alpha):
    from ftd_amd import ftdx
    return ftdx.herk_pol_reduce(ctx, A, N, K, ch, pol, 1, output=out, alpha=alpha)


# samples 320 in all and just past it, in one segment and past it, whole stages of 64 and not
@pytest.mark.parametrize("N,ch", [(256, 2), (385, 2), (520, 2), (256, 350)])
@pytest.mark.parametrize("K,pol", [(160, 2), (161, 2), (200, 2), (256, 2), (320, 2), (336, 2), (128, 4)])
def test_pol_sum_stores_bit_exact(oracle, dev, N, ch, K, pol):
    import torch
    from ftd_amd import ftdx
    B = ch * pol
    qc = oracle.gen_qc_uniform(N + K, N * K * B)
    A = torch.from_numpy(qc).to(dev)
    outs = {}
    for cfg in (-1, 1, 2, 3, 4):
        ctx = ftdx.CutlassComplexGemm()
        ctx.set_launch_config(cfg, -1)
        outs[cfg] = (_pol_sum(ctx, A, N, K, ch, pol, "fp32", 1.0), _pol_sum(ctx, A, N, K, ch, pol, "fp16", 2.0 ** -10))
    torch.cuda.synchronize()
    some = [0, ch - 1]
    per = oracle.herk_int64(qc.reshape(ch, -1)[some].reshape(-1), N, K, len(some) * pol)
    ref = per.reshape(len(some), pol, -1, 2).sum(axis=1)
    for cfg, (c32, c16) in outs.items():
        assert np.array_equal(c32[some].cpu().numpy(), ref.astype(np.float32)), cfg
        assert np.array_equal(c16[some].cpu().numpy(), (ref * 2.0 ** -10).astype(np.float16)), cfg
        assert torch.equal(c32, outs[1][0]) and torch.equal(c16, outs[1][1]), cfg


@pytest.mark.parametrize("fp16", [False, True])
def test_pol_sum_stores_of_large_outputs(dev, fp16):
    """Outputs on both sides of 80 MB: every channel equals the same channel of a small call."""
    import torch
    from ftd_amd import ftdx
    N, K, pol, ch = 520, 256, 2, 160 if fp16 else 80
    out = "fp16" if fp16 else "fp32"
    gen = torch.Generator(device="cpu").manual_seed(1)
    A = torch.randint(0, 256, (ch, pol * N * K), generator=gen, dtype=torch.uint8).to(dev)
    ctx = ftdx.CutlassComplexGemm()
    whole = _pol_sum(ctx, A, N, K, ch, pol, out, 2.0 ** -10)
    assert whole.numel() * whole.element_size() > 80e6
    for c in (0, 1, ch // 2, ch - 1):
        part = _pol_sum(ctx, A[c:c + 1].contiguous(), N, K, 1, pol, out, 2.0 ** -10)
        assert torch.equal(whole[c:c + 1], part), c
