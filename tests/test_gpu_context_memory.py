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
