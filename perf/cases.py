"""Workloads of the domain-wall hot path, for timing and for checking results.

Each case is one call (or one short sequence of calls) that a program built on
this package makes: an application of the Dirac operator, a fermion force, a
Krylov solve or the whole RHMC force.  `listed()` holds the named cases,
`draw()` gives further ones of the same ranges, `prepare()` makes what the
caller has in hand, `run()` is one pass, `work()` the bytes and operations the
pass cannot do without and `exact()` its result in plain 64-bit torch.

Device fields are torch tensors in the library's layouts: FP64 spinors
[rhs][spin][t][y][x][s], FP32 and FP16 spinors [rhs][t][y][x][s][spin] (FP16
with one float scale per site), links [mu][t][y][x].
"""
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "thirring-rhmc_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import confio  # noqa: E402
import thirring_hip as G  # noqa: E402

BETA = 0.3  # theta ~ N(0, 1/beta), the coupling of the benchmark's fields
# The solves run on smooth fields, about the spread of the measurement tests:
# they end within a few hundred iterations, before rounding decides the path
# (on fields of spread beta^-1/2 the iterates of two equally good runs part).
SMOOTH = 0.4
AM3 = 1.0
_stream = None


def listed():
    return [
        # the benchmark's headline: one application of M on the largest lattice
        {"name": "dslash_f64_32x32x32x64", "op": "dslash", "lx": 32, "ly": 32, "lt": 32, "ls": 64,
         "prec": "f64", "dagger": False, "nrhs": 1, "imass": 3},
        # the production generation lattice; Ls = 48 does not divide a wave
        {"name": "dslash_f64_dag_16x16x16x48", "op": "dslash", "lx": 16, "ly": 16, "lt": 16,
         "ls": 48, "prec": "f64", "dagger": True, "nrhs": 1, "imass": 3},
        # the smallest benchmark lattice: launch latency
        {"name": "dslash_f64_8x8x8x8", "op": "dslash", "lx": 8, "ly": 8, "lt": 8, "ls": 8,
         "prec": "f64", "dagger": False, "nrhs": 1, "imass": 1},
        # the batched measurement solves: 16 sources per launch, FP32 Krylov storage
        {"name": "dslash_f32_24x24x24x32_nrhs16", "op": "dslash", "lx": 24, "ly": 24, "lt": 24,
         "ls": 32, "prec": "f32", "dagger": False, "nrhs": 16, "imass": 3},
        # the lowest precision of the mixed solver on the largest lattice
        {"name": "dslash_f16_dag_32x32x32x64", "op": "dslash", "lx": 32, "ly": 32, "lt": 32,
         "ls": 64, "prec": "f16", "dagger": True, "nrhs": 1, "imass": 3},
        # the force terms of every pole of the 25-pole approximation at the production lattice
        {"name": "derivs_batch25_16x16x16x48", "op": "derivs_batch", "lx": 16, "ly": 16, "lt": 16,
         "ls": 48, "npair": 25},
        # one pole's force with the Wilson-kernel operator, odd extents
        {"name": "derivs_wilson_15x15x21x20", "op": "derivs", "lx": 15, "ly": 15, "lt": 21,
         "ls": 20, "kernel": "wilson", "iflag": 0, "imass": 3},
        # the reference's own congrad test lattice, called on its haloed host arrays
        {"name": "congrad_host_12x12x12x24", "op": "congrad", "lx": 12, "ly": 12, "lt": 12,
         "ls": 24, "host": True, "imass": 3, "am": 0.05, "res": 1e-6},
        # the guidance approximation's solve with the secondary (Wilson-kernel) operator, uneven
        # extents
        {"name": "multishift_wilson_14x14x18x20", "op": "multishift", "lx": 14, "ly": 14,
         "lt": 18, "ls": 20, "kernel": "wilson", "nshift": 12, "imass": 3, "am": 0.1,
         "res": 1e-3},
        # the rational-function solve of qmrherm (the Hamiltonian's 25 poles) at the production
        # lattice, FP64 vectors
        {"name": "multishift_f64_16x16x16x48", "op": "multishift", "lx": 16, "ly": 16, "lt": 16,
         "ls": 48, "kernel": "shamir", "nshift": 25, "imass": 3, "am": 0.05, "res": 1e-6},
        # batched measurement sources, each at the poles of an approximation: FP64, then FP32
        # Krylov storage, FP64 correction
        {"name": "solve_mixed_24x24x24x32", "op": "solve", "lx": 24, "ly": 24, "lt": 24, "ls": 32,
         "nsrc": 8, "nshift": 12, "imass": 3, "am": 0.05, "tol": 1e-10, "th32": 1e-2},
        # the whole RHMC force (four rational solves and their derivs) on host arrays
        {"name": "force_host_12x12x12x24", "op": "force", "lx": 12, "ly": 12, "lt": 12, "ls": 24,
         "imass": 3, "am": 0.05, "res": 1e-4},
    ]


def _extents(rng, most, ls_choices):
    """A lattice of at most `most` 5-D sites, x = y as the reference has it in
    two cases of three, sizes even over the logarithm and odd ones among them."""
    ls = rng.choice(ls_choices)
    most4 = most // ls
    v4 = 512.0 * (most4 / 512.0) ** rng.random()
    side = v4 ** (1.0 / 3.0)
    lx = max(4, min(48, int(round(side * 2.0 ** rng.uniform(-0.3, 0.3)))))
    ly = lx if rng.random() < 0.67 else max(4, min(48, lx + rng.randint(-3, 3)))
    lt = max(4, min(64, int(v4 / (lx * ly))))
    return {"lx": lx, "ly": ly, "lt": lt, "ls": ls}


def draw(rng):
    op = rng.choice(["dslash", "dslash", "dslash", "derivs_batch", "derivs", "congrad",
                     "multishift", "solve", "force"])
    imass = rng.choice([1, 3, 3, 3])  # the solves take the generation's imass 3
    if op == "dslash":
        nrhs = rng.choice([1, 1, 2, 4, 7, 12])
        case = _extents(rng, (32 ** 3 * 64) // nrhs, [8, 12, 16, 20, 24, 32, 40, 48, 64])
        case.update(op=op, prec=rng.choice(["f64", "f64", "f32", "f16"]),
                    dagger=rng.random() < 0.5, nrhs=nrhs, imass=rng.choice([imass, imass, 5]))
    elif op == "derivs_batch":
        npair = rng.choice([3, 12, 25])
        case = _extents(rng, 16 ** 3 * 48, [8, 16, 24, 32, 48, 64])
        case.update(op=op, npair=npair)
    elif op == "derivs":
        case = _extents(rng, 24 ** 3 * 32, [8, 12, 16, 20, 32, 48])
        case.update(op=op, kernel=rng.choice(["shamir", "wilson"]), iflag=rng.randint(0, 1),
                    imass=imass)
    elif op == "congrad":
        case = _extents(rng, 16 ** 3 * 24, [12, 16, 20, 24, 32])
        case.update(op=op, host=rng.random() < 0.5, imass=3, am=rng.choice([0.05, 0.1]),
                    res=rng.choice([1e-2, 1e-4, 1e-6]))
    elif op == "multishift":
        case = _extents(rng, 16 ** 3 * 48, [12, 16, 24, 32, 48])
        kernel = rng.choice(["shamir", "shamir", "wilson"])
        case.update(op=op, kernel=kernel, nshift=rng.choice([12, 25]), imass=3,
                    am=rng.choice([0.05, 0.1]) if kernel == "shamir" else 0.1,
                    res=rng.choice([1e-4, 1e-6]) if kernel == "shamir" else 1e-3)
    elif op == "solve":
        case = _extents(rng, 16 ** 3 * 32, [8, 16, 32, 48])
        case.update(op=op, nsrc=rng.choice([1, 4, 12]), nshift=rng.choice([1, 12]), imass=3,
                    am=rng.choice([0.05, 0.1]), tol=1e-10, th32=1e-2)
    else:
        case = _extents(rng, 12 ** 3 * 24, [12, 16, 24])
        case.update(op=op, imass=3, am=rng.choice([0.05, 0.1]), res=1e-4)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dims(case):
    return case["lx"], case["ly"], case["lt"], case["ls"]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 17)


def _gauss(shape, gen):
    """Complex Gaussian noise of unit variance (complex128)."""
    z = torch.randn(tuple(shape) + (2,), dtype=torch.float64, device="cuda", generator=gen)
    return torch.view_as_complex(z.mul_(0.5 ** 0.5))


def _fields(case, seed):
    """theta ([3][t][y][x], float32), its FP64 links (u = 1 + i theta with
    antiperiodic t-links, gauge.F90:12-43) and the generator for the rest."""
    lx, ly, lt, ls = _dims(case)
    gen = _generator(seed)
    spread = SMOOTH if case["op"] in ("congrad", "multishift", "solve", "force") else BETA ** -0.5
    theta = torch.randn((3, lt, ly, lx), device="cuda", generator=gen) * spread
    links = torch.complex(torch.ones_like(theta, dtype=torch.float64), theta.double())
    links[2, lt - 1] *= -1.0
    return theta, links, gen


def _spinors(case, gen, n=1):
    lx, ly, lt, ls = _dims(case)
    return _gauss((n, 4, lt, ly, lx, ls), gen)


def _haloed(v):
    """The reference's haloed Fortran array of a spinor [spin][t][y][x][s] or of
    links [mu][t][y][x]: one periodic cell around every lattice extent."""
    a = v.cpu().numpy()
    a = np.pad(a, [(0, 0)] + [(1, 1)] * (a.ndim - 1), mode="wrap")
    if a.ndim == 5:  # Phi(0:Ls+1, 0:Lx+1, 0:Ly+1, 0:Lt+1, 4)
        return np.asfortranarray(a.transpose(4, 3, 2, 1, 0))
    return np.asfortranarray(a.transpose(3, 2, 1, 0))


def _narrow(psi, prec):
    """An FP64 spinor batch in FP32 or FP16 (+ scales) storage."""
    sites = psi.permute(0, 2, 3, 4, 5, 1).contiguous()
    if prec == "f32":
        return sites.to(torch.complex64), None
    re = torch.view_as_real(sites).float()
    scale = re.abs().amax(dim=(-1, -2))
    return (re / scale[..., None, None]).half().contiguous(), scale.contiguous()


def _poles(n):
    """Shifts and residues of an approximation with n poles: the guidance
    approximation of x^(-1/4) has 12, the Hamiltonian's 25."""
    num, den = confio.remez("remez4g" if n <= 12 else "remez4")[0]
    return np.ascontiguousarray(den[:n]), np.ascontiguousarray(num[1:n + 1])


def prepare(case, seed):
    global _stream
    if _stream is None:
        G.init(0)
        _stream = torch.cuda.Stream()
    theta, links, gen = _fields(case, seed)
    st = {"case": case, "dims": _dims(case), "links": links, "stream": _stream.cuda_stream}
    lx, ly, lt, ls = st["dims"]
    op = case["op"]
    if op == "dslash":
        psi = _spinors(case, gen, case["nrhs"])
        st["am"] = [0.005 * (1 + k) for k in range(case["nrhs"])]
        if case["prec"] == "f64":
            st["in"], st["in_norm"], st["out_norm"] = psi, None, None
        else:
            st["links"] = links.to(torch.complex64)
            st["in"], st["in_norm"] = _narrow(psi, case["prec"])
            st["out_norm"] = None if st["in_norm"] is None else torch.empty_like(st["in_norm"])
        st["out"] = torch.empty_like(st["in"])
    elif op in ("derivs", "derivs_batch"):
        n = case.get("npair", 1)
        st["r"], st["x2"] = _spinors(case, gen, n), _spinors(case, gen, n)
        st["weights"] = [0.37 / (1 + k) for k in range(n)]
        st["flags"] = [k & 1 for k in range(n)]
        st["force"] = torch.empty((3, lt, ly, lx), dtype=torch.float64, device="cuda")
    elif op == "congrad":
        st["phi"], st["guess"] = _spinors(case, gen)[0], _spinors(case, gen)[0]
        if case["host"]:
            for k in ("phi", "guess", "links"):
                st[k] = _haloed(st[k])
        else:
            st["x"] = torch.empty_like(st["guess"])
    elif op == "multishift":
        st["aden"], st["anum"] = _poles(case["nshift"])
        st["phi"] = _spinors(case, gen)[0]
        st["x"] = torch.empty((case["nshift"],) + st["phi"].shape, dtype=torch.complex128,
                              device="cuda")
    elif op == "solve":
        st["links32"] = links.to(torch.complex64)
        st["aden"] = np.zeros(1) if case["nshift"] == 1 else _poles(case["nshift"])[0]
        st["b"] = _spinors(case, gen, case["nsrc"])
        st["x"] = torch.empty((case["nsrc"], case["nshift"]) + st["b"].shape[1:],
                              dtype=torch.complex128, device="cuda")
    else:
        st["phi"], st["links"] = _haloed(_spinors(case, gen)[0]), _haloed(links)
        st["theta"] = np.asfortranarray(theta.cpu().numpy().transpose(3, 2, 1, 0))
        (a4, d4), _ = confio.remez("remez4g")
        (a2, d2), (b2, e2) = confio.remez("remez2g")
        st["coeffs"] = (a4, d4, b2, e2, a2, d2)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case, dims, op = st["case"], st["dims"], st["case"]["op"]
    if op == "dslash":
        G.dslash_dev(st["out"], st["in"], st["links"], dims, st["am"], imass=case["imass"],
                     am3=AM3, dagger=case["dagger"], prec=case["prec"], in_norm=st["in_norm"],
                     out_norm=st["out_norm"], nrhs=case["nrhs"], stream=st["stream"])
        return {"out": st["out"], "norm": st["out_norm"]}
    if op == "derivs":
        with torch.cuda.stream(_stream):
            st["force"].zero_()
        return G.derivs_dev(st["r"], st["x2"], st["weights"][0], case["iflag"], dims, st["force"],
                            am=0.05, imass=case["imass"], kernel=case["kernel"],
                            stream=st["stream"])
    if op == "derivs_batch":
        with torch.cuda.stream(_stream):
            st["force"].zero_()
        return G.derivs_batch_dev(list(st["r"]), list(st["x2"]), st["weights"], st["flags"], dims,
                                  st["force"], stream=st["stream"])
    if op == "congrad":
        if case["host"]:
            x = st["guess"].copy(order="F")
            it, nx = G.congrad(st["phi"], x, st["links"], dims, case["res"], case["am"],
                               case["imass"], am3=AM3)
        else:
            x = st["x"]
            with torch.cuda.stream(_stream):
                x.copy_(st["guess"])
            it, nx = G.congrad_dev(st["phi"], x, st["links"], dims, case["res"], case["am"],
                                   case["imass"], am3=AM3, stream=st["stream"])
        return {"x": x, "itercg": it, "iterations": nx}
    if op == "multishift":
        it, its = G.multishift_dev(st["links"], dims, case["am"], case["imass"], st["aden"],
                                   st["anum"], st["x"], st["phi"], case["res"], 10000, am3=AM3,
                                   kernel=case["kernel"], stream=st["stream"])
        return {"x": st["x"], "iterations": it, "per_shift": its}
    if op == "solve":
        G.multishift_fast_dev(st["links"], st["links32"], dims, case["am"], case["imass"],
                              st["aden"], st["b"], st["x"], tol=case["tol"], maxcg=20000,
                              nsrc=case["nsrc"], th32=case["th32"], am3=AM3, stream=st["stream"])
        return {"x": st["x"]}
    force, its = G.force(st["phi"], case["res"], case["am"], case["imass"], BETA, st["theta"],
                         st["links"], dims, st["coeffs"], am3=AM3)
    return {"force": force, "itercg": np.asarray(its)}


# iterations of the solves at these targets (measured), for the work estimates
_ITERATIONS = {"congrad": 160, "multishift": 240, "solve": 330, "force": 520}


def work(case):
    """Bytes and floating-point operations of one pass: every field read or
    written once per operator application and per vector update."""
    lx, ly, lt, ls = _dims(case)
    v4, v5 = lx * ly * lt, lx * ly * lt * ls
    field, links, op = 64 * v5, 48 * v4, case["op"]
    apply_flops = 4 * 2 * 50 * v5  # 3 spin-projected hops, s hops and mass terms
    if op == "dslash":
        per = {"f64": 64, "f32": 32, "f16": 20}[case["prec"]]
        return {"bytes": case["nrhs"] * 2 * v5 * per + (48 if per == 64 else 24) * v4,
                "flops": case["nrhs"] * apply_flops}
    if op in ("derivs", "derivs_batch"):
        n = case.get("npair", 1)
        return {"bytes": n * 2 * field + 24 * v4, "flops": n * 3 * 160 * v5}
    # a solver iteration: M and M^+ (two fields each) and the r, p, x updates
    n = _ITERATIONS[op] * case.get("nsrc", 1)
    return {"bytes": n * (8 * field + 2 * links), "flops": n * (2 * apply_flops + 100 * v5)}


# ---------------------------------------------------------------------------
# the same results in plain torch, 64 bits
# ---------------------------------------------------------------------------
_GP = ((3, 2, 1, 0), (3, 2, 1, 0), (2, 3, 0, 1))  # (gamma_mu v)[a] = e(mu, a) v[p(mu, a)]
_GE = ((-1j, -1j, 1j, 1j), (-1, 1, 1, -1), (-1j, 1j, 1j, -1j))
_AXIS = (-2, -3, -4)  # x, y, t of [..., spin, t, y, x, s]


def _gamma(mu, v):
    e = torch.tensor(_GE[mu], dtype=v.dtype, device=v.device).reshape(4, 1, 1, 1, 1)
    return e * v[..., list(_GP[mu]), :, :, :, :]


def _hops(v, links, dagger):
    out = torch.zeros_like(v)
    for mu, ax in enumerate(_AXIS):
        u = links[mu][..., None]
        f = u * torch.roll(v, -1, ax)
        b = torch.roll(u.conj() * v, 1, ax)
        d = (f - b) if not dagger else (b - f)
        out -= 0.5 * (f + b) - 0.5 * _gamma(mu, d)
    return out


def _shamir(v, links, am, imass, dagger):
    """M or M^+ (dirac.F90:29-179, 303-494) on spinors [..., spin, t, y, x, s]."""
    up, dn = (slice(0, 2), slice(2, 4)) if dagger else (slice(2, 4), slice(0, 2))
    out = float(np.float32(3.0) - np.float32(AM3) + np.float32(1.0)) * v + _hops(v, links, dagger)
    sp = lambda t, k: t[..., k, :, :, :, :]  # noqa: E731
    sp(out, up)[..., :-1] -= sp(v, up)[..., 1:]
    sp(out, dn)[..., 1:] -= sp(v, dn)[..., :-1]
    m = torch.as_tensor(np.asarray(am, dtype=np.float32).astype(np.float64), device=v.device)
    m = m.reshape(m.shape + (1,) * 4)
    if imass == 5:
        c = -1j if dagger else 1j
        sp(out, up)[..., -1] += c * m * sp(v, dn)[..., -1]
        sp(out, dn)[..., 0] += c * m * sp(v, up)[..., 0]
    else:
        c = 1.0 if imass == 1 else 1j
        sp(out, up)[..., -1] += c * m * sp(v, up)[..., 0]
        sp(out, dn)[..., 0] += (1.0 if imass == 1 else -c) * m * sp(v, dn)[..., -1]
    return out


def _wilson_couplings(v, am, imass, upper_from_below):
    """The s-couplings of the Wilson kernel: two spins take s - 1, the other two
    s + 1, with the mass at the walls (dirac.F90:226-299, 538-625)."""
    m = float(np.float32(am))
    c1, c2 = (-m, -m) if imass == 1 else (-1j * m, 1j * m)
    lo, hi = (slice(0, 2), slice(2, 4)) if upper_from_below else (slice(2, 4), slice(0, 2))
    q = torch.zeros_like(v)
    q[lo][..., 1:] = v[lo][..., :-1]
    q[lo][..., 0] = c1 * v[lo][..., -1]
    q[hi][..., :-1] = v[hi][..., 1:]
    q[hi][..., -1] = c2 * v[hi][..., 0]
    return q


def _wilson(v, links, am, imass, dagger):
    diag = float(np.float32(3.0) - np.float32(AM3))
    slice_op = lambda w: diag * w + _hops(w, links, dagger)  # noqa: E731
    if dagger:
        t = slice_op(v)
        return t + v + _wilson_couplings(t - v, am, imass, False)
    q = _wilson_couplings(v, am, imass, True)
    return slice_op(v + q) + v - q


def _operator(case, links):
    f = _wilson if case.get("kernel") == "wilson" else _shamir
    return lambda v, dag: f(v, links, case["am"], case["imass"], dag)


def _derivs(r, x2, weight, iflag):
    """The force sums of one (R, X2) pair (derivs_module.F90:99-196)."""
    tzi = np.float32(2.0) * np.float32(weight)
    w1, w2 = float(tzi * np.float32(0.5)), float(tzi) * (1.0 if iflag == 0 else -1.0)
    out = []
    for mu, ax in enumerate(_AXIS):
        rf, xf = torch.roll(r, -1, ax), torch.roll(x2, -1, ax)
        wil = (r.conj() * xf).imag - (rf.conj() * x2).imag
        dirac = 0.5 * (r.conj() * _gamma(mu, xf) + rf.conj() * _gamma(mu, x2)).imag
        out.append((w1 * wil + w2 * dirac).sum(dim=(0, -1)))
    return torch.stack(out)


def _norm2(v):
    return float(torch.view_as_real(v).square().sum())


def _congrad(op, phi, x, res):
    """measure_module.F90:9-140."""
    resid = float(np.float32(np.float32(phi.numel()) * np.float32(res)) * np.float32(res))
    x, p, r = x.clone(), x.clone(), phi.clone()
    beta_d = beta_n = 1.0
    for n in range(1, phi.numel()):
        h = op(p, False)
        alpha = beta_n / _norm2(h) if n > 1 else 1.0
        if n > 1:
            x += alpha * p
        r -= alpha * op(h, True)
        beta_n = _norm2(r)
        if beta_n < resid:
            return x
        p = r + (beta_n / beta_d if n > 1 else 0.0) * p
        beta_d = beta_n
    return x


def _multishift(op, aden, corr, b, res, maxcg):
    """multishift_module.F90:71-282; shift i ends at |r_i| corr_i < res."""
    n = len(aden)
    r, p = b.clone(), b.clone()
    x, ps = torch.zeros((n,) + b.shape, dtype=b.dtype, device=b.device), b.repeat(n, 1, 1, 1, 1, 1)
    z1, z2, z3 = np.ones(n), np.ones(n), np.ones(n)
    live, first, last = np.ones(n, bool), 0, n
    delta, om, gam = _norm2(r), 1.0, 0.0
    for _ in range(maxcg):
        h = op(p, False)
        s = op(h, True)
        prev, om = om, -delta / float(torch.sum(torch.view_as_real(p) * torch.view_as_real(s)))
        k = slice(first, last)
        z3[k] = z1[k] * z2[k] * prev / (om * gam * (z1[k] - z2[k])
                                        + z1[k] * prev * (1.0 - aden[k] * om))
        oms = om * z3 / z2
        r += om * s
        lam = _norm2(r)
        gam = lam / delta
        p = r + gam * p
        for i in range(first, last):
            x[i] -= oms[i] * ps[i]
            ps[i] = (gam * z3[i] * oms[i] / (z2[i] * om)) * ps[i] + z3[i] * r
        live &= ~(np.sqrt(delta * z2 * z2) * corr < res)
        if not live.any():
            break
        at = np.flatnonzero(live)
        first, last = at[0], at[-1] + 1
        k = slice(first, last)
        z1[k], z2[k] = z2[k].copy(), z3[k].copy()
        delta = lam
    return x


def exact(case, seed):
    op = case["op"]
    if op == "force":  # four chained solves: over the time that is sensible here
        return None
    _, links, gen = _fields(case, seed)
    if op == "dslash":
        psi = _spinors(case, gen, case["nrhs"])
        am = [0.005 * (1 + k) for k in range(case["nrhs"])]
        if case["prec"] != "f64":
            links = links.to(torch.complex64).to(torch.complex128)
            val, scale = _narrow(psi, case["prec"])
            if scale is None:
                psi = val.to(torch.complex128)
            else:
                psi = torch.view_as_complex((val.double() * scale[..., None, None].double())
                                            .contiguous())
            psi = psi.permute(0, 5, 1, 2, 3, 4)
        out = torch.cat([_shamir(psi[k:k + 1], links, am[k:k + 1], case["imass"], case["dagger"])
                         for k in range(case["nrhs"])])
        if case["prec"] == "f64":
            return {"out": out, "norm": None}
        out = out.permute(0, 2, 3, 4, 5, 1).contiguous()
        if case["prec"] == "f32":
            return {"out": out, "norm": None}
        out = torch.view_as_real(out)
        scale = out.abs().amax(dim=(-1, -2))
        return {"out": out / scale[..., None, None], "norm": scale}
    if op in ("derivs", "derivs_batch"):
        n = case.get("npair", 1)
        r, x2 = _spinors(case, gen, n), _spinors(case, gen, n)
        if op == "derivs_batch":
            return sum(_derivs(r[k], x2[k], 0.37 / (1 + k), k & 1) for k in range(n))
        a, b = r[0], x2[0]
        if case["kernel"] == "wilson":  # derivs_module.F90:41-97, 198-410: the s-couplings
            if case["iflag"] == 1:
                b = b + _wilson_couplings(b, 0.05, case["imass"], True)
            else:  # <R, P X(s')> summed over s: the couplings' adjoint on R
                a = a + _adjoint_couplings(a, 0.05, case["imass"])
        return _derivs(a, b, 0.37, case["iflag"])
    apply = _operator(case, links)
    if op == "congrad":
        x = _congrad(apply, _spinors(case, gen)[0], _spinors(case, gen)[0], case["res"])
        return {"x": _haloed(x) if case["host"] else x, "itercg": None, "iterations": None}
    if op == "multishift":
        aden, anum = _poles(case["nshift"])
        corr = np.abs(anum / aden)
        corr /= np.exp(np.log(corr).mean())
        x = _multishift(apply, aden, corr, _spinors(case, gen)[0], float(np.float32(case["res"])),
                        10000)
        return {"x": x, "iterations": None, "per_shift": None}
    aden = np.zeros(1) if case["nshift"] == 1 else _poles(case["nshift"])[0]
    return {"x": torch.stack([_multishift(apply, aden, np.ones(len(aden)), v,
                                          1e-13 * _norm2(v) ** 0.5, 10000)
                              for v in _spinors(case, gen, case["nsrc"])])}


def _adjoint_couplings(v, am, imass):
    """R'(s') = sum over the couplings (s, s') of conj(c) P R(s)."""
    m = float(np.float32(am))
    c1, c2 = (-m, -m) if imass == 1 else (-1j * m, 1j * m)
    q = torch.zeros_like(v)
    q[:2][..., 1:] = v[:2][..., :-1]
    q[2:][..., :-1] = v[2:][..., 1:]
    q[2:][..., -1] = np.conj(c1) * v[2:][..., 0]
    q[:2][..., 0] = np.conj(c2) * v[:2][..., -1]
    return q
