"""The growth factor's midpoint sums against the plain loop, bit for bit: the
midpoints one rounded addition after the other, the terms and their sum in FP64
in that order (numpy's accumulate is sequential).  Redshifts whose sums start
at, below and above a power of two, below zero and far above the step."""
import numpy as np
import pytest

import simfast21_amd as sf

H0 = 3.24078e-18


def hubble(z, h, om, ol):
    z1 = 1.0 + z
    return h * H0 * np.sqrt(om * z1 * z1 * z1 + ol)


def plain_integral(zz, h, om, ol):
    dz = 0.001
    # a few more than the 1e5 values of the sum, cut where the loop ends
    z = np.add.accumulate(np.concatenate([[zz + dz / 2.0], np.full(100100, dz)]))
    z = z[z < zz + 100.0]
    e = hubble(z, h, om, ol) / hubble(np.float64(0.0), h, om, ol)
    return np.add.accumulate(((1.0 + z) / e / e / e))[-1] * dz


def plain_growth(z, h, om, ol):
    return (hubble(np.float64(z), h, om, ol) / hubble(np.float64(0.0), h, om, ol)
            * plain_integral(z, h, om, ol) / plain_integral(0.0, h, om, ol))


@pytest.mark.parametrize("z", [0.0, 1e-3, 0.0155, 0.9995, 1.0, 7.9996, 9.0, 63.9995, 300.0, -0.3, 1e5])
@pytest.mark.parametrize("h,om,ol", [(0.7, 0.3, 0.7), (0.71, 1.0, 0.0)])
def test_growth_equals_plain_loop(z, h, om, ol):
    _, d, ddt = sf.cosmology(z, h, om, ol, 0.045)
    assert d == plain_growth(z, h, om, ol)
    hi, lo = plain_growth(z + 0.001 / 2, h, om, ol), plain_growth(z - 0.001 / 2, h, om, ol)
    assert ddt == (hi - lo) / 0.001 * (-hubble(np.float64(z), h, om, ol) * (1.0 + z))
