"""The finder's weight table where it does not hold the whole ladder: refilled
before each filter pass, with the bits of a table that does.  A ladder longer
than 1/16 of the card's memory allows (a plane side; a side with separate passes),
and the same ladder with much and with little free memory."""
import gc

import numpy as np
import pytest

import simfast21_amd as sf
from test_gpu_line_batches import boxes, centre_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [96, 256])
def test_long_ladder_equals_its_parts(torch_cuda, n):
    """A ladder's centre map is the cell-wise maximum of its parts' maps."""
    side = 1.5 * n
    a, b = boxes(torch_cuda, n, 60 + n)
    one = (n // 2 + 1) ** 2 * n * 4
    nr = int(torch_cuda.cuda.mem_get_info()[1] / 16 / one) + 2
    radii = list(np.geomspace(0.25 * side, 2.0, nr))
    stats = {}
    w = centre_map(n, side, radii, a, b, stats)
    assert "w_table" in stats
    parts = np.full_like(w, -1)
    for k in range(0, nr, (nr + 2) // 3):
        sub = {}
        np.maximum(parts, centre_map(n, side, radii[k:k + (nr + 2) // 3], a, b, sub), out=parts)
        assert "w_table" not in sub
    assert 0 < (w >= 0).sum() < n ** 3
    assert np.array_equal(w, parts)


@pytest.mark.parametrize("n", [16, 32])
def test_more_radii_than_a_grid_has_planes(torch_cuda, n):
    """65600 radii, five different ones: the map of those five."""
    side = 1.5 * n
    radii = np.geomspace(0.25 * side, 2.0, 5)
    a, b = boxes(torch_cuda, n, 80 + n)
    w = centre_map(n, side, list(radii), a, b)
    assert 0 < (w >= 0).sum() < n ** 3
    assert np.array_equal(centre_map(n, side, list(np.repeat(radii, 13120)), a, b), w)


def test_same_bits_with_little_free_memory(torch_cuda):
    torch = torch_cuda
    n, side, room = 512, 768.0, 85 << 30
    radii = list(np.geomspace(0.25 * side, 2.0, 47))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(12)
    g = 0.5 * torch.randn(n ** 3, generator=gen, device="cuda")
    emis = torch.rand(n ** 3, generator=gen, device="cuda")
    emis *= torch.rand(n ** 3, generator=gen, device="cuda") < 0.3
    got = []
    torch.cuda.empty_cache()
    for full in (False, True):
        gc.collect()
        hold = torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device="cuda") if full else None
        ctx = sf.HiiContext(n, side, radii, sf.INPUT_DIRECT, sf.PATH_FUSED)
        ctx.profile(True)
        x, mean, _ = ctx.diff_forward(g, emis, 1.5)  # P(k)'s FP64 sums go by atomics: last bits vary
        grad, gz, _, _ = ctx.diff_backward(g, emis, 1.5, 0.02, 1.0, np.ones(20))
        assert ("w_table" in ctx.kernel_stats()) == full
        got.append((x.cpu().numpy(), grad.cpu().numpy(), mean, gz))
        ctx.close()
        del hold, x, grad
        torch.cuda.empty_cache()
    assert 0.0 < got[0][2] < 1.0 and np.abs(got[0][1]).max() > 0
    for p, q in zip(*got):
        assert np.array_equal(p, q)
