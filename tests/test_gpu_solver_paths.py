"""Paths of the FP64 reference solvers (measure_module.F90:9-140,
multishift_module.F90:13-284) that the default launch shapes of a small
lattice do not take, and what the solvers leave behind when they stop."""
import numpy as np
import pytest

import dense as D
import oracle as O

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


def test_ring_is_given_back(G):
    """The FP64 multishift's ring of 32 residuals stays in the context, and an
    allocation of the context that fails takes it back (here one of 512 GiB,
    which no card holds and the call reports before any launch)."""
    from hiprt import DeviceArray
    dims = (16, 16, 16, 16)
    lx, ly, lt, ls = dims
    v5 = lx * ly * lt * ls
    rng = np.random.default_rng(52)
    links = np.stack([np.ones(3 * lx * ly * lt), 0.4 * rng.standard_normal(3 * lx * ly * lt)], -1)
    l64 = DeviceArray.from_host(links)
    b, x = DeviceArray.from_host(rng.standard_normal((4 * v5, 2))), DeviceArray((4 * v5, 2), np.float64)
    ring = 32 * 64 * v5
    ctx = G.Context()
    ctx.bind()
    try:
        print("case: ring given back", flush=True)
        G.multishift_dev(l64, dims, 0.1, 3, [0.5], [1.0], x, b, 1e-4, 100)
        assert ctx.scratch_bytes() > ring
        big = (64, 64, 64, 1024)  # 16 GiB fields, 32 shifts
        with pytest.raises(G.ThrError) as e:
            G.multishift_dev(l64, big, 0.1, 3, np.ones(32), np.ones(32), x, b, 1e-4, 100)
        assert e.value.status == G.STATUS["hip"]
        assert ctx.scratch_bytes() - 64 * int(np.prod(big)) < ring
        ctx.trim()
        # and the context still solves
        G.multishift_dev(l64, dims, 0.1, 3, [0.5], [1.0], x, b, 1e-4, 100)
        assert ctx.scratch_bytes() > ring
        ctx.trim()
    finally:
        ctx.unbind()
        ctx.destroy()


# The FP64 multishift's paths: updates once per 32 iterations, with the scalar
# steps as kernels of their own (a march: also the default from 2^18 sites with
# Ls = 32 and 64, from 2^20 with others) and around separate epilogues (Wilson
# kernel, Ls > 64); and updates in every iteration (no ring), behind passes of
# each kind.  Caps inside the first block of 32, at its end, one past it, and in
# the third block.
@pytest.mark.parametrize("path", ["march", "wilson80", "one_site_no_ring", "march_no_ring",
                                  "wilson_no_ring", "wilson80_no_ring"])
@pytest.mark.parametrize("maxcg", [0, 1, 31, 32, 33, 65])
def test_multishift_paths_at_the_cap(G, monkeypatch, maxcg, path):
    """Against the oracle: fewer than 100 iterations on smooth links (spread
    0.4) amplify rounding by less than 1e4, so 1e-11; iteration counts equal."""
    dims = (2, 3, 2, 80) if "80" in path else (3, 5, 4, 12)
    kernel = "wilson" if "wilson" in path else "shamir"
    if "no_ring" in path:
        monkeypatch.setenv("THR_MULTISHIFT_RING", "0")
    if "march" in path:
        G.dslash_set_config(dims, "f64", 2, G.SHAPE_XCD_REMAP)
    rng = np.random.default_rng(53)
    u = O.coef((0.4 * rng.standard_normal(dims[:3] + (3,))).astype(np.float32), dims)
    inp = D.rand_spinor(dims, rng)
    sig = np.array([1e-4, 0.05, 0.7, 9.0])
    print("case: multishift path", path, maxcg, flush=True)
    og, cg, cgs = G.multishift(u, dims, 0.05, 3, sig, np.ones(4), inp, res=1e-5, maxcg=maxcg,
                               kernel=kernel)
    oo, co, cos = O.multishift(u, dims, 0.05, 3, sig, np.ones(4), inp, res=1e-5, maxcg=maxcg,
                               kernel=kernel)
    assert cg == co and np.array_equal(cgs, cos)
    if maxcg == 0:
        assert not og.any()
    else:
        assert np.linalg.norm(og - oo) <= 1e-11 * np.linalg.norm(oo)


def _shamir_80bit(v, u, m, dagger):
    """M or M^+ (imass 3, am3 = 1; dirac.F90:29-179, 303-494) on [spin][t][y][x][s] in
    extended precision."""
    perm, phase = ((3, 2, 1, 0), (3, 2, 1, 0), (2, 3, 0, 1)), ((-1j, -1j, 1j, 1j), (-1, 1, 1, -1),
                                                              (-1j, 1j, 1j, -1j))
    up, dn = (slice(0, 2), slice(2, 4)) if dagger else (slice(2, 4), slice(0, 2))
    out = np.longdouble(3) * v
    for mu in range(3):
        g = np.array(phase[mu], np.clongdouble).reshape(4, 1, 1, 1, 1)
        f = u[mu][..., None] * np.roll(v, -1, -2 - mu)
        b = np.roll(u[mu].conj()[..., None] * v, 1, -2 - mu)
        d = b - f if dagger else f - b
        out -= np.longdouble(0.5) * (f + b - g * d[list(perm[mu])])
    out[up][..., :-1] -= v[up][..., 1:]
    out[dn][..., 1:] -= v[dn][..., :-1]
    out[up][..., -1] += 1j * m * v[up][..., 0]
    out[dn][..., 0] -= 1j * m * v[dn][..., -1]
    return out


def test_multishift_block_sums_are_rounded_at_their_own_size(G):
    """x_i takes the sum of a block's 32 terms in one addition.  A CPU model of
    these solves has a median error of 4.9e-16 of the solution's norm that way,
    and of 7.2e-16 where x_i takes the terms one after another (18 solves of 6
    seeds each); the line lies between, at 6e-16.  Reference: (M^+M + s) x = b
    by CG in 80-bit arithmetic."""
    from hiprt import DeviceArray
    lx, ly, lt, ls = dims = (4, 4, 6, 16)
    sig, errs = np.array([0.3, 0.32, 0.34]), []
    for seed in (61, 62, 63):
        rng = np.random.default_rng(seed)
        u = 1 + 1j * (0.4 * rng.standard_normal((3, lt, ly, lx))).astype(np.float32).astype(float)
        u[2, lt - 1] *= -1
        b = rng.standard_normal((4, lt, ly, lx, ls)) + 1j * rng.standard_normal((4, lt, ly, lx, ls))
        bd = DeviceArray.from_host(np.stack([b.real, b.imag], -1).reshape(-1, 2))
        l64 = DeviceArray.from_host(np.stack([u.real, u.imag], -1).reshape(-1, 2))
        x = DeviceArray((len(sig), b.size, 2), np.float64)
        print("case: block sums of the multishift, seed", seed, flush=True)
        G.multishift_plain_dev(l64, dims, 0.05, 3, sig, bd, x, 1e-16, 4000)
        got = x.to_host()
        ul, m = u.astype(np.clongdouble), np.longdouble(np.float32(0.05))
        for k, s in enumerate(sig):
            want = np.zeros(b.shape, np.clongdouble)
            r = b.astype(np.clongdouble)
            p, rr = r.copy(), (np.abs(r) ** 2).sum()
            r0 = rr
            while rr > np.longdouble(1e-38) * r0:
                q = _shamir_80bit(_shamir_80bit(p, ul, m, False), ul, m, True) + np.longdouble(s) * p
                a = rr / (p.conj() * q).real.sum()
                want += a * p
                r -= a * q
                rn = (np.abs(r) ** 2).sum()
                p, rr = r + (rn / rr) * p, rn
            z = (got[k, :, 0] + 1j * got[k, :, 1]).reshape(b.shape)
            errs.append(float(np.sqrt((np.abs(z - want) ** 2).sum() / (np.abs(want) ** 2).sum())))
    print("errors", " ".join("%.2e" % e for e in errs), flush=True)
    assert np.median(errs) <= 6e-16
