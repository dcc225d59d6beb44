"""ftdx_herk_pol_grid without a forced tile, at the edges of its routes (pipelined kernel, half planes,
fused tile): bit-exact on integer sums against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(N, Ng, seed, cell=2e-3, chan=1):
    """Baselines of antennas whose UV mostly falls on the grid; frequencies; cell size."""
    rng = np.random.default_rng(seed)
    pos = rng.uniform(-0.5, 0.5, (N, 2)) * (0.5 * Ng * cell * 0.2)
    i, j = np.tril_indices(N)
    return (pos[i] - pos[j]).astype(np.float32), np.linspace(0.8e9, 1.4e9, chan), cell


def _reference(oracle, qc, N, K, chan, pols, uv, freqs, Ng, cell):
    """The oracle's grid of qc [chan, pols, N, K]."""
    per = oracle.herk_int64(qc, N, K, chan * pols).reshape(chan, pols, -1, 2).sum(axis=1)
    assert np.abs(per).max() < 2 ** 24
    return oracle.pillbox_grid(per.astype(np.float32), uv, freqs, N * (N + 1) // 2, Ng, chan, cell)


def test_more_segments_than_a_grid_dimension(oracle, dev):
    """70000 polarization segments, past the 65535 input batches that one conversion launch takes: the
    call returns, with the sum of the few segments that are not zero."""
    import torch
    from ftd_amd import ftdx
    N, K, n_pol, Ng = 64, 16, 70000, 64
    full = [0, 1, 35000, 65535, 65536, 69999]
    qc = oracle.gen_qc_uniform(5, N * K * len(full)).reshape(len(full), N, K)
    uv, freqs, cell = _scene(N, Ng, 1)
    A = torch.zeros((n_pol, N, K), dtype=torch.uint8, device=dev)
    A[full] = torch.from_numpy(qc).to(dev)
    grid = torch.zeros((1, Ng, Ng, 2), device=dev)
    uv_d, f_d = torch.from_numpy(uv).to(dev), torch.from_numpy(freqs).to(dev)
    ftdx.herk_pol_grid(ftdx.CutlassComplexGemm(), A, N, K, 1, n_pol, uv_d, f_d, grid, Ng, cell)
    torch.cuda.synchronize()
    ref = _reference(oracle, qc.reshape(-1), N, K, 1, len(full), uv, freqs, Ng, cell)
    assert np.abs(ref).sum() > 0
    assert np.array_equal(grid.cpu().numpy(), ref)


# a tile's waves share its rows at the diagonal and at the edge: one wave's block and parts of 16 rows
# (1, 16, 17, 63 .. 65), blocks without rows (100, 130, 193), whole tiles beside them (256, 300)
@pytest.mark.parametrize("cfg", [-1, 0, 2, 3])
@pytest.mark.parametrize("N", [1, 16, 17, 63, 64, 65, 100, 128, 130, 193, 256, 300])
def test_rows_shared_by_a_tile(oracle, dev, cfg, N):
    """Autocorrelations in one cell (summed over the tile) and in cells of their own, with and without
    a half plane (one baseline per five cells on), on a grid that is not zero."""
    import torch
    from ftd_amd import ftdx
    K, chan, pols = 80, 2, 2
    qc = oracle.gen_qc_uniform(N, N * K * chan * pols)
    ctx = ftdx.CutlassComplexGemm()
    ctx.set_launch_config(cfg, -1)
    A = torch.from_numpy(qc).to(dev)
    for Ng in (33, 700):
        uv, freqs, cell = _scene(N, Ng, N + 1, chan=chan)
        f_d = torch.from_numpy(freqs).to(dev)
        for apart in (False, True):
            if apart:
                d = np.arange(N)
                uv[d * (d + 3) // 2, 0] = (d % 7 - 3) * cell * 0.2
            ref = _reference(oracle, qc, N, K, chan, pols, uv, freqs, Ng, cell)
            grid = torch.full((chan, Ng, Ng, 2), 2.0, device=dev)
            ftdx.herk_pol_grid(ctx, A, N, K, chan, pols, torch.from_numpy(uv).to(dev), f_d, grid, Ng, cell)
            torch.cuda.synchronize()
            assert np.abs(ref).max() < 2 ** 24 - 2
            assert np.array_equal(grid.cpu().numpy(), ref + 2.0), (Ng, apart)


# even and odd grids on both sides of one baseline per eight cells; few inputs with enough channels and not
@pytest.mark.parametrize("N,K,chan,Ng", [(256, 64, 3, 363), (256, 64, 3, 362), (300, 600, 2, 65), (300, 40, 2, 602),
                                         (100, 16, 200, 40), (100, 16, 197, 40), (255, 64, 2, 64)])
def test_half_planes_at_their_line(oracle, dev, N, K, chan, Ng):
    """Baselines on the grid's edge (no mirror cell) and exactly between two cells (rounding away from
    zero is not symmetric about the centre), wavelengths of 1 and 2 m and others."""
    import torch
    from ftd_amd import ftdx
    pols, cell, light = 2, 2e-3, 299792458.0
    qc = oracle.gen_qc_uniform(N + Ng, N * K * chan * pols)
    rng = np.random.default_rng(Ng)
    uv = (rng.integers(-2 * Ng, 2 * Ng + 1, (N * (N + 1) // 2, 2)) * (0.25 * cell)).astype(np.float32)
    d = np.arange(N)
    uv[d * (d + 3) // 2] = 0.0
    freqs = np.resize([light, 0.5 * light, 1.3e9], chan)
    ref = _reference(oracle, qc, N, K, chan, pols, uv, freqs, Ng, cell)
    grid = torch.full((chan, Ng, Ng, 2), 3.0, device=dev)
    ftdx.herk_pol_grid(ftdx.CutlassComplexGemm(), torch.from_numpy(qc).to(dev), N, K, chan, pols,
                       torch.from_numpy(uv).to(dev), torch.from_numpy(freqs).to(dev), grid, Ng, cell)
    torch.cuda.synchronize()
    assert np.abs(ref).max() < 2 ** 24 - 3
    assert np.array_equal(grid.cpu().numpy(), ref + 3.0)


@pytest.mark.parametrize("Ng", [512, 1024])  # 168 MB of half planes; 671 MB, so none
@pytest.mark.parametrize("K", [1008, 1000])
def test_gridding_in_chunks(dev, Ng, K):
    """More channels than one 160 MB chunk of fragment rows: each chunk grids its own channels, at their
    frequencies, into their planes.  Equal to a forced tile's grid, whose sums are exact too (+-1 voltages)."""
    import torch
    from ftd_amd import ftdx
    N, chan, pols = 1024, 120, 2  # 3.1 MB of rows per channel
    gen = torch.Generator(device=dev).manual_seed(K)
    A = torch.tensor([0x11, 0x19, 0x91, 0x99], dtype=torch.uint8, device=dev)[
        torch.randint(0, 4, (chan * pols * N * K,), generator=gen, device=dev)]
    uv, _, cell = _scene(N, Ng, 3)
    uv_d = torch.from_numpy(uv).to(dev)
    freqs = torch.linspace(0.7e9, 1.4e9, chan + 1, dtype=torch.float64, device=dev)
    grids = []
    for cfg in (-1, 0):
        ctx = ftdx.CutlassComplexGemm()
        ctx.set_launch_config(cfg, -1)
        grids.append(torch.zeros((chan, Ng, Ng, 2), device=dev))
        ftdx.herk_pol_grid(ctx, A, N, K, chan, pols, uv_d, freqs, grids[-1], Ng, cell, freq_offset=1)
        torch.cuda.synchronize()
        ctx.close()
    assert float(grids[0].abs().max()) < 2 ** 24
    for c in range(chan):
        assert torch.equal(grids[0][c], grids[1][c]), c
    assert not torch.equal(grids[0][0], grids[0][chan - 1])
