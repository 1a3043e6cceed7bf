"""Sizes of grids and spectra follow their resolution, also when it is changed, and a subclass's
own rings."""
import copy
import pickle

import pytest


@pytest.mark.parametrize("kind", ["OctahedralGaussianGrid", "FullGaussianGrid"])
def test_points_follow_the_rings(sw, kind):
    g = getattr(sw, kind)(1)
    for n in (1, 2, 3, 24, 47):
        g.nlat_half = n
        assert g.npoints == sum(g.nlons) == getattr(sw, kind)(n).npoints
        assert copy.copy(g).npoints == pickle.loads(pickle.dumps(g)).npoints == g.npoints


def test_points_of_a_subclass(sw):
    class Reduced(sw.grids._RingGrid):
        def __init__(self, n, step):
            super().__init__(n)
            self.step = step

        def nlon_ring(self, j):
            return 20 + self.step * j
    assert Reduced(3, 8).npoints == 2 * (20 + 28 + 36)


def test_harmonics_follow_the_truncation(sw):
    s = sw.Spectrum(33, 32)
    assert s.nharm == len(s.degrees_orders()[0])
    s.lmax, s.mmax = 22, 21
    assert s.nharm == len(s.degrees_orders()[0]) == sw.Spectrum(22, 21).nharm
