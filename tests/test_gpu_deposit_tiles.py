"""The displacement deposit on grids of more tiles than blocks, each block taking
several, against an FP64 deposit in numpy: whole tiles (256) and partial ones at
the end of every axis (212); displacements that stay near, that carry a part of
the grid along, and that scatter too far for a tile's sums."""
import numpy as np
import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu
H, OM, OL = 0.7, 0.3, 0.7


def cic64(m, pos, value):
    """auxiliary.c:761-808 in FP64 (pos as the kernel's float32 positions)."""
    cell = np.trunc(pos)
    far = pos - cell
    cell = np.where(far < 0, cell - 1, cell).astype(np.int64)
    far = np.abs(far)
    grid = np.zeros(m ** 3)
    for c in range(8):
        up = [(c >> k) & 1 for k in range(3)]
        w = value
        for k in range(3):
            w = w * (far[k] if up[k] else 1 - far[k])
        at = [(cell[k] + up[k]) % m for k in range(3)]
        grid += np.bincount(((at[0] * m + at[1]) * m + at[2]).ravel(), w.ravel(), m ** 3)
    return grid.reshape(m, m, m)


@pytest.mark.parametrize("m,amp,shift", [(256, 1.1, 0.0), (212, 1.1, 0.0), (212, 0.7, 11.0), (256, 40.0, 0.0)])
def test_displacement_of_many_tiles(torch_cuda, m, amp, shift):
    """shift: an eighth of the grid moves by that many cells as well."""
    torch = torch_cuda
    rng = np.random.default_rng(m + int(amp))
    L_h, z = 1.0 * m, 9.0
    p = dict(hubble=H, omega_m=OM, omega_b=0.045, omega_lambda=OL, box_len=L_h, n=m, n_halo=m)
    g_in = sf.cosmology(300.0, H, OM, OL)[1]
    g = sf.cosmology(z, H, OM, OL)[1] - g_in
    vscale = np.float32(m / L_h * H)
    v = []
    for _ in range(3):
        a = amp * rng.standard_normal((m, m, m))
        a[: m // 2, : m // 2, m // 2:] += shift
        v.append((a / (vscale * g)).astype(np.float32))
    d0 = rng.standard_normal((m, m, m)).astype(np.float32)
    ctx = sf.HiiContext(m, L_h, [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=m)
    box = torch.empty(m ** 3, dtype=torch.float32, device="cuda")
    dev = [torch.from_numpy(a.ravel()).cuda() for a in (*v, d0)]
    idx = np.meshgrid(*(np.arange(m, dtype=np.float64),) * 3, indexing="ij", sparse=True)
    # the float32 product, then one rounding of its multiple plus the cell: left
    # of the border a cell's weights jump at whole positions, so an ulp counts
    pos = [((v[k] * vscale).astype(np.float64) * float(np.float32(g)) + idx[k]).astype(np.float32)
           .astype(np.float64) for k in range(3)]
    ref = cic64(m, pos, 1 + d0.astype(np.float64) * g_in) - 1.0
    # an FP32 position of up to m + 6 amp + shift cells is off by half an ulp in
    # the product and in the sum: that moves the far weight of masses near 1, of
    # which about eight meet in a cell (plus FP32 sums of the same size)
    tol = 8 * 2 * (m + 6 * amp + shift) * 2.0 ** -23
    for rep in range(2):
        box.fill_(7.0)
        ctx.nldensity(p, z, *dev, box_halo=box)
        got = box.cpu().numpy().reshape(m, m, m)
        assert np.abs(got - ref).max() <= tol, (rep, np.abs(got - ref).max(), tol)
    ctx.close()


@pytest.mark.parametrize("n,m,offset", [(20, 40, 0), (20, 40, 1), (20, 41, 0), (7, 24, 0), (33, 67, 1),
                                        (70, 140, 0), (70, 70, 0)])
def test_block_average(torch_cuda, n, m, offset):
    """The averages against the same compensated FP32 sums in numpy, exactly:
    blocks of 1 to 3 cells, even and odd grids, a grid off its alignment."""
    torch = torch_cuda
    torch.manual_seed(m)
    p = dict(hubble=H, omega_m=OM, omega_b=0.045, omega_lambda=OL, box_len=1.0 * m, n=n, n_halo=m)
    v = [20 * torch.randn(m ** 3, device="cuda") for _ in range(3)]
    ctx = sf.HiiContext(n, 1.0 * m, [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=m)
    box = torch.empty(m ** 3 + 1, device="cuda")[offset:offset + m ** 3]
    out, _ = ctx.nldensity(p, 9.0, *v, torch.randn(m ** 3, device="cuda"), box_halo=box)
    ctx.close()
    g = box.cpu().numpy().reshape(m, m, m)
    sm = int(np.floor(np.float32(m) / n + 0.5))
    sm -= 1 if n * sm > m else 0
    total = np.zeros((n, n, n), np.float32)
    comp = np.zeros_like(total)
    for a, b, c in np.ndindex(sm, sm, sm):
        y = g[a:n * sm:sm, b:n * sm:sm, c:n * sm:sm] - comp
        t = total + y
        comp = (t - total) - y
        total = t
    ref = total * (np.float32(1) / (np.float32(sm) * sm * sm))
    assert np.array_equal(out.cpu().numpy().reshape(n, n, n), ref)
