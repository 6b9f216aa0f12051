"""Names of Dslash launch shapes, through the C entry points that need no GPU:
the pair that get_config reports selects the same kernel when it is pinned."""
import ctypes

import pytest

import thirring_hip as G

MARCH_FLAGS = 2 | 4 | 16 | 64 | 128 | 256


@pytest.fixture(autouse=True)
def unpinned():
    G.dslash_clear_config()
    yield
    G.dslash_clear_config()


def get(dims, prec, nrhs=1):
    tc, fl = ctypes.c_int(), ctypes.c_int()
    assert G.lib().thr_dslash_get_config_nrhs(G._dims(dims), G.PREC[prec], nrhs, ctypes.byref(tc),
                                              ctypes.byref(fl)) == 0
    return tc.value, fl.value


def put(dims, prec, tc, fl):
    return G.lib().thr_dslash_set_config(G._dims(dims), G.PREC[prec], tc, fl)


def one_site(pair):
    return pair[0] == 1 and pair[1] & MARCH_FLAGS == G.SHAPE_ONE_SITE


# small launches, and FP32 and FP16 ones of every size off Ls = 32 and 64
@pytest.mark.parametrize("dims,prec", [((4, 4, 4, 8), "f64"), ((16, 16, 16, 48), "f64"),
                                       ((8, 8, 8, 64), "f16"), ((32, 32, 32, 48), "f32")])
def test_one_site_default_is_restored(dims, prec):
    saved = get(dims, prec)
    assert one_site(saved) and saved[1] < 256
    assert put(dims, prec, 2, 32) == 0
    assert get(dims, prec) == (2, 32)
    assert put(dims, prec, *saved) == 0
    assert get(dims, prec) == saved


def test_march_default_is_restored():
    dims = (32, 32, 32, 64)
    for prec in ("f64", "f32", "f16"):
        saved = get(dims, prec)
        assert not one_site(saved)
        assert put(dims, prec, *saved) == 0 and get(dims, prec) == saved


def test_every_other_pair_still_marches():
    """Each pair of the defined flags reads back as it was pinned; the one-site
    kernel is one setting of the march's flags, at t-chunk 1 only."""
    dims = (4, 4, 4, 64)
    for tc in (1, 2):
        for fl in range(512):
            assert put(dims, "f64", tc, fl) == 0
            assert get(dims, "f64") == (tc, fl)
    assert put(dims, "f64", 1, 512) == 1 and put(dims, "f64", 1, 1024) == 1


def test_clear_unpins_both_batch_classes():
    dims = (8, 8, 8, 64)
    single, batch = get(dims, "f64"), get(dims, "f64", 32)
    assert one_site(single) and not one_site(batch)
    other = get((4, 4, 4, 8), "f64")
    assert put(dims, "f64", 3, 1) == 0 and put((4, 4, 4, 8), "f64", 2, 1) == 0
    assert get(dims, "f64", 32) == (3, 1)
    assert G.lib().thr_dslash_clear_config(G._dims(dims), 0) == 0
    assert (get(dims, "f64"), get(dims, "f64", 32)) == (single, batch)
    assert get((4, 4, 4, 8), "f64") == (2, 1)
    G.dslash_clear_config()
    assert get((4, 4, 4, 8), "f64") == other
    assert G.lib().thr_dslash_clear_config(G._dims((4, 0, 4, 8)), 0) == 1
    assert G.lib().thr_dslash_clear_config(G._dims(dims), 3) == 1


# the environment's settings take effect on launches whose default is the
# one-site kernel, too: those that only the march reads select it
@pytest.mark.parametrize("name,value,want", [
    ("TCHUNK", "3", (3, 0)), ("UNIFORM", "1", (1, 2)), ("LANESHIFT", "0", (1, 0)),
    ("LDSX", "1", (1, 16)), ("LDSY", "1", (1, 256)), ("OCC", "2", (1, 128))])
def test_environment_selects_the_march(monkeypatch, name, value, want):
    dims = (4, 4, 6, 12)
    assert one_site(get(dims, "f64"))
    monkeypatch.setenv("THR_DSLASH_" + name, value)
    tc, fl = get(dims, "f64")
    assert (tc, fl & MARCH_FLAGS) == want
    monkeypatch.setenv("THR_DSLASH_SITE", "1")
    assert one_site(get(dims, "f64"))


@pytest.mark.parametrize("name,bit", [("REMAP", 1), ("BOXES", 8), ("NT", 32)])
def test_environment_settings_of_both_kernels(monkeypatch, name, bit):
    for dims in ((4, 4, 6, 12), (32, 32, 32, 64)):
        was = get(dims, "f64")
        monkeypatch.setenv("THR_DSLASH_" + name, "0" if was[1] & bit else "1")
        assert get(dims, "f64") == (was[0], was[1] ^ bit)
        monkeypatch.delenv("THR_DSLASH_" + name)
