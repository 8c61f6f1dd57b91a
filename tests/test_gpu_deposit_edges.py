"""Deposits at their edges: the displacement deposit where a tile's targets fit
the block's LDS, where they scatter too far for it, on grids smaller than a
tile, at remainders of the tile and across the periodic border; the catalog
deposit where blocks are one cell, several, and do not divide the grid.  FP64
references in numpy."""
import numpy as np
import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu
H, OM, OL = 0.7, 0.3, 0.7


def cic(grid, pos, value):
    """auxiliary.c:761-808 in FP64 (pos as the kernel's float32 positions)."""
    m = grid.shape[0]
    cell = np.trunc(pos)
    far = pos - cell
    cell = np.where(far < 0, cell - 1, cell).astype(np.int64)
    far = np.abs(far)
    for c in range(8):
        up = [(c >> k) & 1 for k in range(3)]
        w = value.copy()
        for k in range(3):
            w = w * (far[k] if up[k] else 1 - far[k])
        np.add.at(grid, tuple((cell[k] + up[k]) % m for k in range(3)), w)


@pytest.mark.parametrize("m,amp", [(5, 0.3), (16, 1.0), (33, 0.0), (40, 2.0), (48, 60.0), (70, 3.0)])
def test_displacement(torch_cuda, m, amp):
    """amp: displacement in cells (0: every cell stays; 60: targets anywhere)."""
    torch = torch_cuda
    rng = np.random.default_rng(m)
    L_h, z = 1.0 * m, 9.0
    p = dict(hubble=H, omega_m=OM, omega_b=0.045, omega_lambda=OL, box_len=L_h, n=m, n_halo=m)
    g_in = sf.cosmology(300.0, H, OM, OL)[1]
    g = sf.cosmology(z, H, OM, OL)[1] - g_in
    vscale = np.float32(m / L_h * H)
    v = [(amp / (vscale * g) * rng.standard_normal((m, m, m))).astype(np.float32) for _ in range(3)]
    d0 = rng.standard_normal((m, m, m)).astype(np.float32)
    ctx = sf.HiiContext(m, L_h, [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=m)
    box = torch.empty(m ** 3, dtype=torch.float32, device="cuda")
    out, _ = ctx.nldensity(p, z, *(torch.from_numpy(a.ravel()).cuda() for a in v),
                           torch.from_numpy(d0.ravel()).cuda(), box_halo=box)
    ctx.close()
    idx = np.meshgrid(*(np.arange(m, dtype=np.float64),) * 3, indexing="ij")
    pos = np.stack([(v[k].astype(np.float64) * float(vscale) * g + idx[k]).astype(np.float32).astype(np.float64)
                    for k in range(3)])
    ref = np.full((m, m, m), -1.0)
    cic(ref, pos, 1 + d0.astype(np.float64) * g_in)
    got = box.cpu().numpy().reshape(m, m, m)
    # an FP32 position of up to m + 3 amp cells is off by half an ulp in the
    # product and in the sum: that moves the far weight of masses near 1, of
    # which about eight meet in a cell (plus FP32 sums of the same size)
    tol = 8 * 2 * (m + 6 * amp) * 2.0 ** -23
    assert np.abs(got - ref).max() <= tol, (m, amp, np.abs(got - ref).max(), tol)
    assert np.array_equal(out.cpu().numpy().reshape(m, m, m), got)  # n = n_halo: blocks of one cell


@pytest.mark.parametrize("n,m", [(20, 20), (20, 40), (16, 50), (7, 24), (30, 64)])
def test_catalog(torch_cuda, n, m):
    torch = torch_cuda
    rng = np.random.default_rng(n * m)
    L_h, z, count = 1.0 * m, 8.0, 4000
    mass = 10 ** rng.uniform(8.0, 10.5, count)
    pos = rng.uniform(0, m, (count, 3))
    pos[:3] = [[0.0, 0.0, 0.0], [m - 0.25, 3.5, m - 1.0], [-0.3, 2.2, 1.0]]
    pos[3:1000] = pos[3]  # many halos in one cell
    cat = np.column_stack([mass, pos]).astype(np.float32)
    ctx = sf.HiiContext(n, L_h, [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=m)
    out, mean = ctx.sfrd(torch.from_numpy(cat).cuda(), z)
    empty, mean0 = ctx.sfrd(torch.zeros((0, 4), device="cuda"), z)
    ctx.close()
    c = cat.astype(np.float64)
    qion = 10.0 ** (2.05707274e-02 * z + 5.29944413e+01)
    rate = 1.575e39 * (1 + z) ** 2.27044695 / qion * c[:, 0] * (c[:, 0] / 9.367608e+07) ** 0.44 \
        * np.exp(-(9.367608e+07 / c[:, 0]) ** 3)
    grid = np.zeros((m, m, m))
    cic(grid, c[:, 1:].T, rate)
    sm = int(np.floor(np.float32(m) / n + 0.5))
    sm -= 1 if n * sm > m else 0
    g = grid[: n * sm, : n * sm, : n * sm].reshape(n, sm, n, sm, n, sm).mean((1, 3, 5)) / (L_h / m) ** 3
    got = out.cpu().numpy().astype(np.float64).reshape(n, n, n)
    # per halo: powf, expf and five products (a few ulp each); sums in FP64
    assert np.all(np.abs(got - g) <= 16 * 2.0 ** -23 * g + 1e-30), np.abs(got - g).max() / g.max()
    assert abs(mean - g.mean()) <= 16 * 2.0 ** -23 * g.mean()
    assert float(empty.abs().max()) == 0.0 and mean0 == 0.0
