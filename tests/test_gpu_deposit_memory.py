"""Catalog deposits whose FP64 sums do not fit the device memory: refused with
SF21_ERR_ALLOC, never added up in fewer bits."""
import gc

import pytest

import simfast21_amd as sf

pytestmark = pytest.mark.gpu


def test_sums_that_do_not_fit(torch_cuda):
    """Each context's 2048^3 sums take 64 GiB: contexts until one is refused."""
    torch = torch_cuda
    gc.collect()
    torch.cuda.empty_cache()
    n, z = 2048, 8.0
    halo = torch.tensor([[1e9, 3.3, 4.4, 5.5]], device="cuda")
    out = torch.empty(n ** 3, device="cuda")
    contexts, first = [], None
    fits = True
    while fits:
        contexts.append(sf.HiiContext(n, float(n), [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=2 * n))
        fits = torch.cuda.mem_get_info()[0] >= 8 * n ** 3
        print(f"context {len(contexts)}: fits {fits}", flush=True)
        if fits:
            contexts[-1].sfrd(halo, z, out=out)
            corner = out[: 4 * n * n].clone()
            first = corner if first is None else first
            assert torch.equal(corner, first) and float(first.max()) > 0
    with pytest.raises(sf.Sf21Error) as e:
        contexts[-1].sfrd(halo, z, out=out)
    assert e.value.code == sf.SF21_ERR_ALLOC
    # the refused context works once there is room
    contexts.pop(0).close()
    contexts[-1].sfrd(halo, z, out=out)
    assert torch.equal(out[: 4 * n * n], first)
    for c in contexts:
        c.close()
    del out
    torch.cuda.empty_cache()


def test_one_cell_blocks_take_no_sums(torch_cuda):
    torch = torch_cuda
    n = 512
    halo = torch.tensor([[1e9, 3.3, 4.4, 5.5]], device="cuda")
    out = torch.empty(n ** 3, device="cuda")
    c = sf.HiiContext(n, float(n), [], sf.INPUT_HALO, sf.PATH_DEPOSIT, n_halo=n)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    c.halo_emissivity(halo, 8.0, out=out)
    assert float(out.max()) > 0 and before - torch.cuda.mem_get_info()[0] < 8 * n ** 3
    c.close()
