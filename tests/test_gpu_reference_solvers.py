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
