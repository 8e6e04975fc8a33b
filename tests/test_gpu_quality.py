"""The reduced gauge quality on lattices of few blocks (the block that ends
last reduces) and of more (a second kernel): the sum of the per-site values
within the rounding of its tree, MAX exactly their largest, and the same bits
from every call, also on one handle in turns with another lattice's check."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 1 block; 72.2; exactly 256 (the last size of few blocks); 257.25; 1065.5 (more than the 1024 partial sums)
@pytest.mark.parametrize("dims", [(2, 2, 4, 6), (6, 10, 14, 22), (16, 16, 16, 16), (14, 14, 14, 24), (20, 22, 22, 28)])
@pytest.mark.parametrize("kernels", ["LandauKernelsSU3", "MAGKernelsSU3", "U1xU1KernelsSU3"])
@pytest.mark.parametrize("dtype", ["F64", "F32"])
def test_reduced_quality_is_the_sum_of_the_sites(gf, gpu, dtype, kernels, dims):
    lat = gf.Lattice(dims, getattr(gf, dtype))
    V = int(np.prod(dims))
    d = gf.DeviceBuffer(lat.nbytes)
    gf.CommonKernelsSU3(lat).setHot(V, 1, d, None, 5, 1)
    K = getattr(gf, kernels)
    st = gf.GaugeFixingStats(K, d, lat)
    st_max = gf.GaugeFixingStats(K, d, lat, crit=gf.CRIT_MAX)
    seen = set()
    for _ in range(4):
        st.generateGaugeQuality()
        st_max.generateGaugeQuality()
        assert st_max.getCurrentGff() == st.getCurrentGff()
        seen.add((st.getCurrentGff(), st.getCurrentA(), st_max.getCurrentA()))
    assert len(seen) == 1
    gff, theta, theta_max = seen.pop()

    dg, da = gf.DeviceBuffer(8 * V), gf.DeviceBuffer(8 * V)
    K(lat).generateGaugeQualityPerSite(V, 1, d, dg, da)
    g, a = dg.download(np.float64), da.download(np.float64)
    # a block's tree (8 levels), up to 2 partials in a row, a tree of 10 levels, two scalings
    eps = 32 * 2.0 ** -53
    assert abs(gff - math.fsum(g) / 12 / V) <= eps * np.abs(g).sum() / 12 / V
    assert abs(theta - math.fsum(a) / 3 / V) <= eps * np.abs(a).sum() / 3 / V
    assert theta_max == a.max() * (1.0 / 3.0)
