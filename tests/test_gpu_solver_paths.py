"""Paths of the FP64 reference solvers (measure_module.F90:9-140,
multishift_module.F90:13-284) that the default launch shapes of a small
lattice do not take, and what the solvers leave behind when they stop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import thirring_hip as G
    G.init(0)
    return G


# alpha = |r|^2 / |M p|^2 is 0 / 0 in the second iteration of a solve whose
# squares all underflow (a target of 0 lets the first one pass).  The passes
# carry the scalar steps on small launches and with the Wilson kernel; a pinned
# march runs them as kernels of their own.
@pytest.mark.parametrize("path", ["one_site", "march", "wilson", "noalloc"])
def test_congrad_stopped_by_alpha_leaves_x(G, path):
    from hiprt import DeviceArray
    dims = (4, 4, 6, 16) if path != "march" else (4, 6, 6, 16)
    lx, ly, lt, ls = dims
    rng = np.random.default_rng(51)
    links = np.stack([np.ones(3 * lx * ly * lt), 0.4 * rng.standard_normal(3 * lx * ly * lt)], -1)
    l64 = DeviceArray.from_host(links)
    x0 = 1e-170 * rng.standard_normal((4 * lx * ly * lt * ls, 2))
    phi, x = DeviceArray.from_host(np.zeros_like(x0)), DeviceArray.from_host(x0)
    if path == "march":
        G.dslash_set_config(dims, "f64", 2, G.SHAPE_XCD_REMAP)
    print("case: congrad stopped by alpha", path, flush=True)
    with pytest.raises(G.ThrNonFinite):
        if path == "noalloc":
            G.congrad_dev_noalloc(phi, x, l64, dims, 0.0, 0.1, 3, niterc=50)
        else:
            G.congrad_dev(phi, x, l64, dims, 0.0, 0.1, 3, niterc=50,
                          kernel="wilson" if path == "wilson" else "shamir")
    assert np.array_equal(x.to_host(), x0)
