"""Every launch choice that the autotuner searches, forced, against the default's
centre map and box, on the sides that run the column and row passes (256: 16
values per thread exist; 192: 8 only).  The choices regroup the same per-line
work, so map, box and mean are equal bit for bit."""
import numpy as np
import pytest

import simfast21_amd as sf
from test_gpu_autotune import tune_key
from test_gpu_line_batches import boxes

pytestmark = pytest.mark.gpu


def slice_of(n, side, radii, a, b, **kw):
    ctx = sf.HiiContext(n, side, radii, sf.INPUT_DIRECT, sf.PATH_FUSED, **kw)
    x, mean = ctx.run_slice(a, b)
    got = x.cpu().numpy(), mean, np.asarray(ctx.weight_map()).copy(), ctx.tuning()
    ctx.close()
    return got


def check(torch, tmp_path, monkeypatch, n, ct, cw, rw, fp, tile, K):
    side = 1.5 * n
    radii = list(np.geomspace(0.25 * side, 2.0, 11))
    a, b = boxes(torch, n, 500 + n)
    monkeypatch.delenv("SF21_TUNE_CACHE", raising=False)
    x0, m0, w0, _ = slice_of(n, side, radii, a, b)
    assert 0 < (w0 >= 0).sum() < n ** 3
    arch = torch.cuda.get_device_properties(0).gcnArchName.split(":")[0]
    cache = tmp_path / "tune.txt"
    cache.write_text(f"{tune_key(arch, n, side, radii)} | tile={tile} K={K} ct={ct} cw={cw} rw={rw} "
                     f"fp={fp} | 0.0 ms\n")
    monkeypatch.setenv("SF21_TUNE_CACHE", str(cache))
    x1, m1, w1, t = slice_of(n, side, radii, a, b)
    assert (t["cols_tile"], t["cols_wide"], t["rows_wide"], t["filter_pair"], t["filter_tile"],
            t["radius_batch"]) == (ct, cw, rw, fp, tile, K)
    assert np.array_equal(w0, w1) and np.array_equal(x0, x1) and m0 == m1


# K = 3, 4: the ladder of 11 is no multiple; filter tile 4 comes by setting only
@pytest.mark.parametrize("ct,cw,rw,fp,tile,K", [
    (8, 0, 0, 0, 16, 11), (16, 0, 1, 0, 8, 4), (16, 2, 0, 1, 16, 3), (16, 1, 1, 1, 8, 11),
    (16, 3, 0, 0, 16, 4), (32, 1, 1, 1, 16, 3), (32, 3, 0, 1, 8, 11), (32, 0, 1, 0, 16, 11),
    (16, 1, 0, 0, 4, 5)])
def test_256(torch_cuda, tmp_path, monkeypatch, ct, cw, rw, fp, tile, K):
    check(torch_cuda, tmp_path, monkeypatch, 256, ct, cw, rw, fp, tile, K)


@pytest.mark.parametrize("ct,cw,fp,tile,K", [
    (8, 0, 0, 16, 11), (16, 2, 1, 8, 4), (16, 0, 1, 16, 3), (32, 0, 0, 8, 11), (16, 0, 0, 4, 5)])
def test_192(torch_cuda, tmp_path, monkeypatch, ct, cw, fp, tile, K):
    check(torch_cuda, tmp_path, monkeypatch, 192, ct, cw, 0, fp, tile, K)


def test_512_defaults_and_tuned_choice(torch_cuda, tmp_path, monkeypatch):
    """The largest side: 16-value row pass and 32 prefetching columns."""
    check(torch_cuda, tmp_path, monkeypatch, 512, 32, 3, 1, 0, 16, 4)
