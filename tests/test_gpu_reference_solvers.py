"""Edges of the FP64 reference solvers (multishift_module.F90:13-284,
measure_module.F90:9-140) on the GPU against the oracle.

Tolerances: a solve of k < 100 iterations on smooth fields (theta spread 0.4)
amplifies rounding by less than 1e4, so two correct orders of summation agree
to 1e-11; iteration counts are equal."""
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


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def smooth(dims, seed):
    rng = np.random.default_rng(seed)
    th = (0.4 * rng.standard_normal(dims[:3] + (3,))).astype(np.float32)
    return rng, O.coef(th, dims)


# iterations around the 32-iteration blocks of the shift updates: a cap inside
# the first block, at its end, one past it, and in the third block
@pytest.mark.parametrize("kernel", ["shamir", "wilson"])
@pytest.mark.parametrize("maxcg", [0, 1, 31, 32, 33, 65])
def test_multishift_blocks_at_the_cap(G, maxcg, kernel):
    dims = (3, 5, 4, 12)
    rng, u = smooth(dims, 31)
    inp = D.rand_spinor(dims, rng)
    sig = np.array([1e-4, 0.05, 0.7, 9.0])
    print("case: multishift cap", maxcg, kernel, flush=True)
    # the heavier shifts converge inside a block and leave the window
    og, cg, cgs = G.multishift(u, dims, 0.05, 3, sig, np.ones(4), inp, res=1e-5, maxcg=maxcg,
                               kernel=kernel)
    oo, co, cos = O.multishift(u, dims, 0.05, 3, sig, np.ones(4), inp, res=1e-5, maxcg=maxcg,
                               kernel=kernel)
    assert cg == co and np.array_equal(cgs, cos)
    if maxcg == 0:
        assert not og.any()
    else:
        assert rel(og, oo) <= 1e-11


@pytest.mark.parametrize("n", [1, 25, 32])
def test_multishift_shift_counts(G, n):
    """One shift, the 25 of the rational approximation, the most allowed."""
    dims = (4, 4, 6, 8)
    rng, u = smooth(dims, 32)
    inp = D.rand_spinor(dims, rng)
    sig = np.geomspace(1e-3, 60.0, n)
    num = np.geomspace(0.01, 3.0, n)
    print("case: multishift shifts", n, flush=True)
    og, cg, cgs = G.multishift(u, dims, 0.1, 3, sig, num, inp, res=1e-6, maxcg=500)
    oo, co, cos = O.multishift(u, dims, 0.1, 3, sig, num, inp, res=1e-6, maxcg=500)
    assert cg == co and np.array_equal(cgs, cos)
    assert rel(og, oo) <= 1e-11


def test_wilson_congrad_after_a_larger_shamir_solve(G):
    """The Wilson kernel's epilogue fills fewer partial sums than the next sum
    takes: what a Shamir solve on another lattice left there must not count."""
    big, dims = (8, 8, 8, 16), (4, 4, 8, 8)
    rng, ub = smooth(big, 33)
    G.congrad(D.rand_spinor(big, rng), D.rand_spinor(big, rng), ub, big, res=1e-2, am=0.05, imass=3)
    rng, u = smooth(dims, 34)
    phi = D.rand_spinor(dims, rng)
    xg, xo = np.zeros_like(phi), np.zeros_like(phi)
    print("case: wilson congrad after shamir", flush=True)
    g = G.congrad(phi, xg, u, dims, res=1e-3, am=0.1, imass=3, kernel="wilson")
    o = O.congrad(phi, xo, u, dims, res=1e-3, am=0.1, imass=3, kernel="wilson")
    assert g == o
    assert rel(O.interior(xg), O.interior(xo)) <= 1e-10


# s-lines in segments of 1, 4, 16, 32 and 64 lanes, filled and part filled;
# Ls = 80 takes the kernel that walks the slice pairs
@pytest.mark.parametrize("dims", [(4, 3, 2, 1), (3, 5, 4, 4), (5, 3, 4, 12), (3, 3, 5, 20),
                                  (4, 5, 3, 48), (2, 3, 3, 64), (3, 2, 3, 80)])
@pytest.mark.parametrize("iflag", [0, 1])
@pytest.mark.parametrize("imass", [1, 3])
def test_derivs_wilson_lines(G, imass, iflag, dims):
    """The sums have 8 Ls terms of equal size: 1e-12 as for the Shamir force."""
    rng = np.random.default_rng(35)
    R, X2 = D.rand_spinor(dims, rng), D.rand_spinor(dims, rng)
    base = np.asfortranarray(rng.standard_normal(dims[:3] + (3,)))
    print("case: derivs wilson", dims, imass, iflag, flush=True)
    a = dict(kernel="wilson", am=0.3, imass=imass)
    dg = G.derivs(R, X2, 0.37, iflag, dims, base.copy(order="F"), **a)
    do = O.derivs(R, X2, 0.37, iflag, dims, base.copy(order="F"), **a)
    assert rel(dg - base, do - base) <= 1e-12


@pytest.mark.parametrize("dims", [(4, 3, 2, 1), (3, 5, 4, 4), (5, 3, 4, 12), (3, 3, 5, 20),
                                  (4, 5, 3, 48), (2, 3, 3, 64), (3, 2, 3, 80)])
@pytest.mark.parametrize("imass", [1, 3])
def test_dslash_wilson_lines(G, imass, dims):
    """The Wilson-kernel operator on the same line lengths, to the Dslash tolerance 1e-13."""
    rng, u = smooth(dims, 36)
    r = D.rand_spinor(dims, rng)
    print("case: dslash wilson", dims, imass, flush=True)
    for g, o in ((G.dslash, O.dslash), (G.dslashd, O.dslashd)):
        a = g(r, u, dims, 0.3, imass, kernel="wilson")
        b = o(r, u, dims, 0.3, imass, kernel="wilson")
        assert rel(O.interior(a), O.interior(b)) <= 1e-13


@pytest.mark.parametrize("dims", [(14, 14, 3, 20), (3, 5, 4, 4), (3, 2, 3, 80)])
def test_congrad_wilson_lines(G, dims):
    """The fused epilogues of the Wilson kernel (more blocks than the Shamir
    grid at 14 x 14 x 20) and, above Ls = 64, the separate ones."""
    rng, u = smooth(dims, 37)
    phi = D.rand_spinor(dims, rng)
    xg, xo = np.zeros_like(phi), np.zeros_like(phi)
    print("case: congrad wilson", dims, flush=True)
    g = G.congrad(phi, xg, u, dims, res=1e-2, am=0.2, imass=3, kernel="wilson")
    o = O.congrad(phi, xo, u, dims, res=1e-2, am=0.2, imass=3, kernel="wilson")
    assert g == o
    assert rel(O.interior(xg), O.interior(xo)) <= 1e-11


# one site per thread (the default of small launches): lines of every
# remainder, blocks that end inside a slab, lattices the XCD boxes do and do
# not divide
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (3, 5, 2, 1), (2, 2, 2, 2), (5, 3, 7, 12), (4, 4, 4, 48),
                                  (8, 8, 8, 8), (3, 5, 4, 70), (4, 2, 8, 64)])
@pytest.mark.parametrize("imass", [1, 3, 5])
def test_dslash_one_site_per_thread(G, imass, dims):
    """FP64 to the Dslash tolerance 1e-13; FP32 and FP16 fields against the
    FP64 result to 2e-6 and 4e-3 (one rounding per stored number, as
    test_device_precisions), two right-hand sides of different mass."""
    from hiprt import DeviceArray
    rng, u = smooth(dims, 38)
    v5 = int(np.prod(dims))
    am = np.array([0.05, 0.3], dtype=np.float32)
    r = [D.rand_spinor(dims, rng) for _ in am]
    xh = np.stack([D.interior_vec(a) for a in r])  # (2, 4 V5) spin planes
    lin = u[1:-1, 1:-1, 1:-1, :].reshape(-1, order="F")
    l64 = DeviceArray.from_host(np.stack([lin.real, lin.imag], axis=-1))
    l32 = DeviceArray.from_host(np.stack([lin.real, lin.imag], axis=-1).astype(np.float32))
    ri = np.stack([xh.real, xh.imag], axis=-1)  # (2, 4 V5, 2)
    sites = ri.reshape(2, 4, v5, 2).transpose(0, 2, 1, 3)
    scale = np.abs(sites).max(axis=(2, 3)).astype(np.float32)
    print("case: one site per thread", dims, imass, flush=True)
    for dagger, of in ((False, O.dslash), (True, O.dslashd)):
        ref = np.stack([D.interior_vec(of(a, u, dims, float(m), imass)) for a, m in zip(r, am)])
        out = DeviceArray(ri.shape, np.float64)
        G.dslash_dev(out, DeviceArray.from_host(ri), l64, dims, am, imass=imass, dagger=dagger,
                     nrhs=2)
        got = out.to_host()
        assert rel(got[..., 0] + 1j * got[..., 1], ref) <= 1e-13
        refs = np.stack([ref.real, ref.imag], -1).reshape(2, 4, v5, 2).transpose(0, 2, 1, 3)
        out = DeviceArray(sites.shape, np.float32)
        G.dslash_dev(out, DeviceArray.from_host(np.ascontiguousarray(sites).astype(np.float32)), l32,
                     dims, am, imass=imass, dagger=dagger, prec="f32", nrhs=2)
        assert rel(out.to_host().astype(np.float64), refs) <= 2e-6
        q = DeviceArray.from_host(np.ascontiguousarray((sites / scale[..., None, None])
                                                       .astype(np.float16)))
        out, on = DeviceArray(sites.shape, np.float16), DeviceArray(scale.shape, np.float32)
        G.dslash_dev(out, q, l32, dims, am, imass=imass, dagger=dagger, prec="f16", nrhs=2,
                     in_norm=DeviceArray.from_host(scale), out_norm=on)
        got = out.to_host().astype(np.float64) * on.to_host()[..., None, None]
        assert rel(got, refs) <= 4e-3


# congrad's batches poll after 4, 12, 28, 60, ... iterations: caps inside a
# batch, at its end and one past it, with the passes carrying the scalar steps
# (24: small launch) and as launches of their own (a pinned shape)
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("niterc", [0, 1, 2, 4, 5, 12, 13, 30])
def test_congrad_batches_at_the_cap(G, niterc, pinned):
    dims = (4, 4, 6, 24) if not pinned else (4, 6, 4, 24)
    rng, u = smooth(dims, 39)
    phi, x0 = D.rand_spinor(dims, rng), D.rand_spinor(dims, rng)
    if pinned:
        G.dslash_set_config(dims, "f64", 2, G.SHAPE_XCD_REMAP)
    xg, xo = x0.copy(order="F"), x0.copy(order="F")
    print("case: congrad cap", niterc, pinned, flush=True)
    g = G.congrad(phi, xg, u, dims, res=1e-9, am=0.1, imass=3, niterc=niterc)
    o = O.congrad(phi, xo, u, dims, res=1e-9, am=0.1, imass=3, niterc=niterc)
    assert g == o
    assert rel(O.interior(xg), O.interior(xo)) <= 1e-11


# the marching kernel (32 < Ls <= 64, Lx % 4 == 0): whole groups of 8 pairs and
# pairs left over, more than one launch of 32 pairs, t chunks with a remainder;
# and the one-step kernel with a block count that is no multiple of 8
@pytest.mark.parametrize("dims,npair", [((4, 3, 5, 33), 3), ((4, 3, 5, 48), 9), ((8, 6, 21, 64), 40),
                                        ((3, 5, 3, 20), 33), ((16, 16, 9, 40), 32)])
def test_derivs_batch_splits(G, dims, npair):
    """Against the single derivs of each pair, summed: the same terms in another
    order of additions, 1e-13 of the sum's norm."""
    from hiprt import DeviceArray
    lx, ly, lt, ls = dims
    rng = np.random.default_rng(40)
    nsp = 4 * lx * ly * lt * ls
    few = [DeviceArray.from_host(rng.standard_normal((nsp, 2))) for _ in range(6)]
    rs = [few[k % 6] for k in range(npair)]
    xs = [few[(k + 1 + k // 6) % 6] for k in range(npair)]
    an, fl = 0.1 + rng.random(npair), [k % 2 for k in range(npair)]
    base = rng.standard_normal(3 * lx * ly * lt)
    one, all_ = DeviceArray.from_host(base), DeviceArray.from_host(base)
    print("case: derivs batch splits", dims, npair, flush=True)
    for k in range(npair):
        G.derivs_dev(rs[k], xs[k], an[k], fl[k], dims, one)
    G.derivs_batch_dev(rs, xs, an, fl, dims, all_)
    assert rel(all_.to_host(), one.to_host()) <= 1e-13


# one site per thread (a remainder, one shift), the t march on whole lines
# (2^18 sites in a batch) and off them (more than 2^20)
@pytest.mark.parametrize("dims,nsrc,n", [((3, 5, 4, 12), 3, 1), ((5, 3, 7, 32), 2, 3),
                                         ((16, 16, 16, 32), 2, 2), ((13, 5, 22, 64), 3, 1),
                                         ((17, 16, 21, 47), 4, 1)])
def test_true_residuals_of_any_x(G, nsrc, n, dims):
    """|b - (M^+M + sigma_i) x_i| / |b| of random b and x against the oracle's
    operator: no cancellation, sums of positive terms, so rounding only (1e-13
    as the operator's own tolerance)."""
    from hiprt import DeviceArray
    rng, u = smooth(dims, 40)
    v5 = int(np.prod(dims))
    am = np.array([0.05, 0.3, 0.01, 0.1][:nsrc], dtype=np.float32)
    sig = np.array([0.02, 1.5, 0.3][:n])
    c = rng.standard_normal((nsrc, n + 1, 4 * v5, 2))
    print("case: true residuals", dims, nsrc, n, flush=True)
    lin = u[1:-1, 1:-1, 1:-1, :].reshape(-1, order="F")
    l64 = DeviceArray.from_host(np.stack([lin.real, lin.imag], axis=-1))
    got = G.true_residuals_dev(l64, dims, am, 3, sig,
                               DeviceArray.from_host(np.ascontiguousarray(c[:, 0])),
                               DeviceArray.from_host(np.ascontiguousarray(c[:, 1:])), nsrc=nsrc)
    z = c[..., 0] + 1j * c[..., 1]
    for k in range(nsrc):
        for i in range(n):
            a = O.dirac_op_shifted(D.from_vec(z[k, 1 + i], dims), u, dims, float(am[k]), 3,
                                   shift=sig[i])
            want = np.linalg.norm(z[k, 0] - D.interior_vec(a)) / np.linalg.norm(z[k, 0])
            assert abs(got[k, i] - want) <= 1e-13 * want


@pytest.mark.parametrize("tc,flags", [(1, 6), (2, 22), (3, 55), (4, 256 | 22)])
@pytest.mark.parametrize("imass", [1, 3, 5])
def test_dslash_f16_lines_of_64(G, imass, tc, flags):
    """The FP16 march with a wave per s-line (scalar links and lane moves, with
    and without the exchanges along x and y), where the s hops and the wall
    terms go around the wave: against the oracle to 4e-3, and each end of the
    line by itself, to 4e-3 of that slice."""
    from hiprt import DeviceArray
    dims = (4, 6, 5, 64)
    rng, u = smooth(dims, 41)
    v5 = int(np.prod(dims))
    r = D.rand_spinor(dims, rng)
    v = D.interior_vec(r)
    sites = np.stack([v.real, v.imag], -1).reshape(4, v5, 2).transpose(1, 0, 2)
    scale = np.abs(sites).max(axis=(1, 2)).astype(np.float32)
    lin = u[1:-1, 1:-1, 1:-1, :].reshape(-1, order="F")
    l32 = DeviceArray.from_host(np.stack([lin.real, lin.imag], axis=-1).astype(np.float32))
    q = DeviceArray.from_host(np.ascontiguousarray((sites / scale[:, None, None])
                                                   .astype(np.float16)))
    out, on = DeviceArray(sites.shape, np.float16), DeviceArray(scale.shape, np.float32)
    saved = G.dslash_get_config(dims, "f16")
    print("case: FP16 lines of 64", imass, tc, flags, flush=True)
    try:
        G.dslash_set_config(dims, "f16", tc, flags)
        for dagger, of in ((False, O.dslash), (True, O.dslashd)):
            w = D.interior_vec(of(r, u, dims, 0.3, imass))
            ref = np.stack([w.real, w.imag], -1).reshape(4, v5, 2).transpose(1, 0, 2)
            G.dslash_dev(out, q, l32, dims, 0.3, imass=imass, dagger=dagger, prec="f16",
                         in_norm=DeviceArray.from_host(scale), out_norm=on)
            got = out.to_host().astype(np.float64) * on.to_host()[:, None, None]
            assert rel(got, ref) <= 4e-3
            for s in (0, 63):
                assert rel(got[s::64], ref[s::64]) <= 4e-3
    finally:
        G.dslash_set_config(dims, "f16", *saved)
