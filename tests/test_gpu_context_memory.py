"""Device memory that a context holds, against the sizes of what its path
reads.  Allocations are whole pages: 64 MiB are left for that."""
import numpy as np
import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu
SLACK = 64 << 20


def held(torch, n, radii, path=sf.PATH_FUSED, **kw):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ctx = sf.HiiContext(n, 1.5 * n, radii, sf.INPUT_DIRECT, path, **kw)
    now = torch.cuda.mem_get_info()[0]
    ctx.close()
    return before - now


def ladder(n, nr):
    return list(np.geomspace(0.3 * n, 2.0, nr))


def test_plain_path_holds_its_own_weights_only(torch_cuda):
    """A radius adds its FP64-rounded weights per integer |k|^2, nothing else."""
    n, few, many = 256, 2, 47
    held(torch_cuda, n, ladder(n, few), sf.PATH_PLAIN)  # first use of the library
    per_radius = 4 * (3 * (n // 2) ** 2 + 1)
    grown = held(torch_cuda, n, ladder(n, many), sf.PATH_PLAIN) - \
        held(torch_cuda, n, ladder(n, few), sf.PATH_PLAIN)
    assert grown <= (many - few) * per_radius + SLACK, grown / 2 ** 20


def test_plain_path_filtered_pair(torch_cuda):
    """The inspection hook of a plain context gives the fused path's pair."""
    torch = torch_cuda
    n = 128
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    a, b = (torch.rand(n ** 3, generator=g, device="cuda") for _ in range(2))
    pairs = []
    for path in (sf.PATH_PLAIN, sf.PATH_FUSED):
        ctx = sf.HiiContext(n, 1.5 * n, ladder(n, 5), sf.INPUT_DIRECT, path)
        pairs.append(ctx.filtered(a, b, radius_index=3))
        ctx.close()
    assert torch.equal(*pairs)


@pytest.mark.parametrize("K", [1, 3, 1000])
def test_radius_batch_bounds_a_line_side(torch_cuda, K):
    """On a side without a register plan radius_batch bounds the pairs and the
    weights; the slice stays the same."""
    torch = torch_cuda
    n, nr = 240, 40
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    a = torch.exp(0.8 * torch.randn(n ** 3, generator=g, device="cuda"))
    b = torch.exp(1.2 * torch.randn(n ** 3, generator=g, device="cuda") - 0.3)
    b *= torch.rand(n ** 3, generator=g, device="cuda") < 0.3
    got = []
    for k in (0, K):
        ctx = sf.HiiContext(n, 1.5 * n, ladder(n, nr), sf.INPUT_DIRECT, sf.PATH_FUSED, radius_batch=k)
        x, mean = ctx.run_slice(a, b)
        got.append((x, mean, np.asarray(ctx.weight_map()).copy()))
        ctx.close()
    assert torch.equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
    assert np.array_equal(got[0][2], got[1][2]) and 0 < (got[0][2] >= 0).sum() < n ** 3
    # pairs and at most as much for the weights, the spectrum, two integer maps
    held(torch, n, ladder(n, 2))
    bound = (2 * min(K, nr) + 2) * 8 * n ** 3 + SLACK
    assert held(torch, n, ladder(n, nr), radius_batch=K) <= bound


def test_automatic_batch_makes_room_for_stored_fields(torch_cuda):
    """The finder's automatic batch gives its memory back where the
    differentiable mode's stored fields would otherwise not fit."""
    torch = torch_cuda
    torch.cuda.empty_cache()
    n = 256
    pair, total = 8 * n ** 3, torch.cuda.mem_get_info()[1]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    g = 0.5 * torch.randn(n ** 3, generator=gen, device="cuda")
    emis = torch.rand(n ** 3, generator=gen, device="cuda")
    # automatic storage: fields of 0.36 of the memory fit half of what 16 pairs
    # leave free, and not half of what a third of the memory leaves
    nr = int(0.36 * total / pair)
    ctx = sf.HiiContext(n, 1.5 * n, ladder(n, nr), sf.INPUT_DIRECT, sf.PATH_FUSED)
    assert ctx.radius_batch > 100
    ctx.diff_backward(g, emis, 1.5, 0.02, 1.0, None)
    ctx.profile(True)
    ctx.diff_backward(g, emis, 1.5, 0.02, 1.0, None)
    # one sweep of filter passes: the second reads the stored fields
    assert ctx.kernel_stats()["filter_i"][0] == (nr + 15) // 16
    ctx.close()
    # storage asked for: 0.8 of the memory
    ctx = sf.HiiContext(n, 1.5 * n, ladder(n, int(0.8 * total / pair)), sf.INPUT_DIRECT, sf.PATH_FUSED)
    assert ctx.radius_batch > 100
    ctx.diff_store_fields(1)
    assert ctx.radius_batch == 16
    ctx.close()
