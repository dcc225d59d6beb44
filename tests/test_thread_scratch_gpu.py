"""Scratch of the stateless entry point (a context per thread) goes back."""
import threading
import time

import pytest

pytestmark = pytest.mark.gpu

N, K, B = 2048, 2048, 4  # the pipelined kernel's: 25 MB of rows


def _call(torch, ftdx, A, C):
    ftdx.herk_int4(A, N, K, B, C=C)
    torch.cuda.synchronize()


def test_a_threads_scratch_goes_back_at_its_end(dev):
    import torch
    from ftd_amd import ftdx
    A = torch.full((N * K * B,), 0x11, dtype=torch.uint8, device=dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    _call(torch, ftdx, A, C)
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(8):
        t = threading.Thread(target=_call, args=(torch, ftdx, A, C))
        t.start()
        t.join()
    for _ in range(50):  # a thread's end follows its join
        lost = free0 - torch.cuda.mem_get_info()[0]
        if lost < 20e6:
            break
        time.sleep(0.1)
    assert lost < 20e6, lost
    assert bool((C[..., 0] == 2.0 * K).all())


def test_end_herk_without_a_context(dev):
    import torch
    from ftd_amd import ftdx
    A = torch.full((N * K * B,), 0x11, dtype=torch.uint8, device=dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)
    _call(torch, ftdx, A, C)
    free0 = torch.cuda.mem_get_info()[0]
    assert ftdx.lib().ftdx_end_herk(None) == ftdx.FTDX_OK
    assert torch.cuda.mem_get_info()[0] - free0 > 20e6
    assert ftdx.lib().ftdx_end_herk(None) == ftdx.FTDX_OK
    C.zero_()
    _call(torch, ftdx, A, C)
    assert bool((C[..., 0] == 2.0 * K).all())


@pytest.mark.parametrize("N,K,B,rows", [(512, 1024, 20, False), (256, 4000, 12, False), (2048, 2048, 4, True)])
def test_init_herk_reserves_what_the_call_uses(dev, N, K, B, rows):
    """Fragment rows only for shapes that the pipelined kernel runs; their first call allocates nothing."""
    import torch
    from ftd_amd import ftdx
    A = torch.full((N * K * B,), 0x11, dtype=torch.uint8, device=dev)
    C = torch.zeros((B, N * (N + 1) // 2, 2), device=dev)

    def call(c):
        assert c.herk(A, C, N, K, B, input=ftdx.InputPrecision.INT4, output=ftdx.OutputPrecision.FP32, tune=False) == 0
        torch.cuda.synchronize()

    first = ftdx.CutlassComplexGemm()  # the runtime's own allocations for these kernels
    call(first)
    first.close()
    C.zero_()
    ctx = ftdx.CutlassComplexGemm()
    free0 = torch.cuda.mem_get_info()[0]
    ctx.init_herk(N, K, B)
    free1 = torch.cuda.mem_get_info()[0]
    assert (free0 - free1 > 10e6) == rows and free0 - free1 >= 0
    call(ctx)
    assert torch.cuda.mem_get_info()[0] == free1
    assert bool((C[..., 0] == 2.0 * K).all())
