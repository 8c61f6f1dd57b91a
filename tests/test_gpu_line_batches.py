"""Batches of radii on box sides without a register plan: one run of a ladder
against runs of its parts.

A cell's entry in the centre map is the squared reach of the largest radius
whose centre test it passes, and a radius' test does not depend on the other
radii, so the map of a ladder is the cell-wise maximum of the maps of its parts,
exactly.  Sides: 24 and 120 (plane by plane, an odd number of 8-plane groups),
144 (the first with separate passes), 200 (lines shared by two planes, a block
count that is no multiple of 8), 576 (several batches); and a ladder whose
weight table is refilled per batch."""
import os

import numpy as np
import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu


def boxes(torch, n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rec = torch.exp(0.8 * torch.randn(n ** 3, generator=g, device="cuda"))
    ion = torch.exp(1.2 * torch.randn(n ** 3, generator=g, device="cuda") - 0.3)
    ion *= torch.rand(n ** 3, generator=g, device="cuda") < 0.3
    return rec, ion


def centre_map(n, side, radii, a, b, stats=None):
    ctx = sf.HiiContext(n, side, radii, sf.INPUT_DIRECT, sf.PATH_FUSED)
    if stats is not None:
        ctx.profile(True)
    ctx.run_slice(a, b)
    w = np.asarray(ctx.weight_map()).copy()
    if stats is not None:
        stats.update(ctx.kernel_stats())
    ctx.close()
    return w


# 64, 96 and 128 have a plan: their plane pass splits a ladder over blocks by
# the room in LDS (one block a CU at 96 and 128)
@pytest.mark.parametrize("n,nr", [(24, 9), (120, 11), (144, 7), (200, 7), (576, 14),
                                  (64, 27), (96, 31), (96, 2), (128, 9)])
def test_ladder_equals_its_parts(torch_cuda, n, nr):
    side = 1.5 * n
    radii = list(np.geomspace(0.25 * side, 2.0, nr))
    a, b = boxes(torch_cuda, n, 40 + n)
    w = centre_map(n, side, radii, a, b)
    parts = np.full_like(w, -1)
    for k in range(0, nr, 3):
        np.maximum(parts, centre_map(n, side, radii[k:k + 3], a, b), out=parts)
    assert 0 < (w >= 0).sum() < n ** 3
    assert np.array_equal(w, parts)


def test_block_orders_of_shared_lines(torch_cuda, tmp_path, monkeypatch):
    torch = torch_cuda
    n, side = 200, 300.0
    radii = [40.0, 6.0, 2.0]
    a, b = boxes(torch, n, 77)
    cache = tmp_path / "tune.txt"
    ctx = sf.HiiContext(n, side, radii, sf.INPUT_DIRECT, sf.PATH_FUSED)
    x0 = ctx.run_slice(a, b)[0].clone()
    ctx.autotune(a, b, cache_path=cache)
    ctx.close()
    key = cache.read_text().split("|")[0].strip()
    monkeypatch.setenv("SF21_TUNE_CACHE", str(cache))
    for mask in (0, 2, 4, 6):
        with open(cache, "a") as f:
            f.write(f"{key} | gx={mask} | 1.000 ms\n")
        c = sf.HiiContext(n, side, radii, sf.INPUT_DIRECT, sf.PATH_FUSED)
        assert c.line_order == mask
        assert torch.equal(c.run_slice(a, b)[0], x0), mask
        c.close()


def test_weight_table_refilled_per_batch(torch_cuda):
    """A table of more than 1/16 of the free memory is kept for one batch."""
    n, side = 400, 600.0
    a, b = boxes(torch_cuda, n, 91)
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
    assert np.array_equal(w, parts)
