"""What a user of the engine has it do, as cases that can be timed and compared.

A case is one call (or one pair of calls) of `pynfam_amd.engine.GpuEngine` on a
seeded synthetic HFB solution with HFBTHO's block structure (`synthetic.py`).
The basis and the operator are the handle a program builds once and keeps; the
seed makes what changes from call to call: the contour (its upper end, as
another nucleus' Q value would set it), the amplitudes or the densities.

`kind` of a case:
  solve        a batch of contour points to convergence (max_iter 300, si < 1e-7)
  restart      a batch interrupted after six iterations and continued from its
               stored amplitudes, residuals and strengths
  hamiltonian  calc_hamiltonian, the plug-in boundary of the reference's ifam
  transforms   qp2sp and sp2qp, the block transforms on either side of it
Sizes: nsh oscillator shells, ngh x ngl Gauss-Hermite x Gauss-Laguerre points.
"""
import functools
import math

import numpy as np

# (Z, N, beta2) by the shells of the basis
NUCLEI = {"light": (20, 28, 0.0), "rare-earth": (60, 92, 0.3), "heavy": (70, 120, 0.25)}
OPERATORS = [("F", 0), ("GT", 0), ("GT", 1), ("R", 0), ("R", 1), ("P", 0), ("P", 1), ("RS0", 0), ("RS1", 0),
             ("RS1", 1), ("RS2", 0), ("RS2", 1), ("RS2", 2), ("PS0", 0)]
COUPLINGS = dict(vpair_t0=-346.352, override_cs0=128.279, override_csr=0.0, override_cds=0.0)
PRECISIONS = {"fp64": 0, "mixed": 1, "mixed-norefine": 2}
ITERATIONS = 11          # iterations of a contour point, on average over the batches below


def _case(name, kind, nucleus, nsh, ngh, ngl, op, K, npts=1, precision="fp64", **kw):
    return dict(name=name, kind=kind, nucleus=nucleus, nsh=nsh, ngh=ngh, ngl=ngl, op=op, K=K, npts=npts,
                precision=precision, hist64=bool(kw.get("hist64", False)), want_x=bool(kw.get("want_x", False)),
                cross=bool(kw.get("cross", False)))


def listed():
    return [
        # one point per process, as pynfam launches pnfam_main: the amplitudes
        # come back for the .bin file.  A small basis, then the production one.
        _case("point-n8", "solve", "light", 8, 40, 40, "GT", 0, 1, want_x=True),
        _case("point-n16", "solve", "rare-earth", 16, 40, 40, "GT", 1, 1, want_x=True),
        # whole contours of one operator-K: a small and odd one, the archived
        # runs' 30 points, the benchmark's 128 points, a few on the largest basis
        _case("contour-n7", "solve", "light", 7, 23, 19, "GT", 1, 13),
        _case("contour-n12", "solve", "rare-earth", 12, 40, 40, "GT", 0, 30),
        _case("contour-n16", "solve", "rare-earth", 16, 40, 40, "GT", 0, 128),
        _case("contour-n20", "solve", "heavy", 20, 50, 50, "GT", 1, 12),
        # a first-forbidden set with its cross-terms on the device, amplitudes
        # returned as the rate calculation wants them
        _case("forbidden-n10", "solve", "rare-earth", 10, 31, 33, "R", 1, 24, want_x=True, cross=True),
        # the mixed-precision path: the benchmark's batch with the FP64 history
        # it sets, and a small batch with the defaults
        _case("mixed-n16", "solve", "rare-earth", 16, 40, 40, "GT", 0, 128, "mixed", hist64=True),
        _case("mixed-n12", "solve", "rare-earth", 12, 40, 40, "GT", 1, 20, "mixed"),
        # an interrupted batch continued from its stored amplitudes
        _case("restart-n10", "restart", "rare-earth", 10, 32, 32, "GT", 0, 8),
        # the engine inside the reference's own iteration: host arrays in and out
        _case("hamiltonian-n16", "hamiltonian", "rare-earth", 16, 40, 40, "GT", 0),
        _case("transforms-n16", "transforms", "rare-earth", 16, 40, 40, "GT", 1),
    ]


def draw(rng):
    """A case of the same ranges: bases of 6 to 18 shells, grids of 16 to 50
    points each way (odd ones too), 1 to 128 points, every operator."""
    kind = rng.choice(["solve"] * 5 + ["restart", "hamiltonian", "transforms"])
    nsh = rng.randint(6, 18)
    nucleus = rng.choice(["light", "rare-earth"]) if nsh < 10 else rng.choice(["rare-earth", "heavy"])
    lo = 16 if nsh < 10 else 30
    ngh, ngl = rng.randint(lo, 50), rng.randint(lo, 50)
    op, K = rng.choice(OPERATORS[:3] * 3 + OPERATORS[3:])
    # points: within the work of 128 points at 16 shells on the 40 x 40 grid
    room = 128.0 * (16.0 / nsh) ** 5 * 1600.0 / (ngh * ngl)
    most = max(1.0, min(128.0, 0.5 * room))
    if kind == "restart":
        most = min(most, 16.0)
    npts = int(round(math.exp(rng.uniform(0.0, math.log(most))))) if most > 1 else 1
    precision = "fp64"
    if kind == "solve":
        precision = rng.choice(["fp64", "fp64", "mixed", "mixed-norefine"])
    c = _case("", kind, nucleus, nsh, ngh, ngl, op, K, npts if kind in ("solve", "restart") else 1, precision,
              hist64=rng.random() < 0.5 and precision != "fp64", want_x=kind == "solve" and npts <= 8,
              cross=kind == "solve" and op not in ("F", "GT") and rng.random() < 0.5)
    del c["name"]
    return c


# ---- what a program has in hand ----------------------------------------------
@functools.lru_cache(maxsize=2)
def _problem(nucleus, nsh, ngh, ngl, op, K):
    from pynfam_amd.problem import build_problem
    from pynfam_amd.synthetic import synthetic_basis
    Z, N, beta = NUCLEI[nucleus]
    basis = synthetic_basis(Z=Z, N=N, n00=nsh, beta=beta, ngh=ngh, ngl=ngl)
    return build_problem(basis, op, K, "-", "SKOP", **COUPLINGS)


def _prob(case):
    return _problem(case["nucleus"], case["nsh"], case["ngh"], case["ngl"], case["op"], case["K"])


_held = {}          # the one engine a program keeps over its batches: {key: engine}


def _engine(case):
    from pynfam_amd.crossterms import crossterm_problems
    from pynfam_amd.engine import GpuEngine
    key = tuple(case[k] for k in ("nucleus", "nsh", "ngh", "ngl", "op", "K", "precision", "hist64", "cross"))
    if key not in _held:
        for e in _held.values():
            e.close()
        _held.clear()
        prob = _prob(case)
        eng = GpuEngine(prob)
        if case["precision"] != "fp64":
            eng.set_option("mix_hist64", 1 if case["hist64"] else 0)
        if case["cross"]:
            eng.set_crossterms([p.f_elem for _, p in crossterm_problems(prob, **COUPLINGS)])
        _held[key] = eng
    return _held[key]


def _contour(prob, npts, rng):
    """The computed half of a closed contour around [0, E]; E below the window
    of the lowest two-quasiparticle energies, as the Q values of a chain vary."""
    from pynfam_amd.rate import circle_contour, eqrpa_max_beta_minus
    sols = prob.basis.sols
    e = eqrpa_max_beta_minus(sols[0].ala, sols[1].ala) * rng.uniform(0.8, 1.0)
    return np.asarray(circle_contour(0.0, e, 2 * npts)["z"][:npts])


def _amplitudes(prob, rng):
    """Amplitudes of one frequency, ReX, ImX, ReY, ImY: of the size the Green's
    function gives them, falling with the two-quasiparticle energy."""
    scale = np.exp(rng.uniform(-4.0, 0.0, prob.nxy))
    return [rng.standard_normal(prob.nxy) * scale for _ in range(4)]


def prepare(case, seed):
    rng = np.random.default_rng([seed, case["nsh"], case["npts"]])
    prob, eng = _prob(case), _engine(case)
    state = {"case": case, "engine": eng}
    if case["kind"] == "solve":
        state["omega"] = _contour(prob, case["npts"], rng)
    elif case["kind"] == "restart":
        w = _contour(prob, case["npts"], rng)
        r = eng.solve(w, max_iter=6, want_x=True)
        state.update(omega=w, stored={"x": r["x"], "si": r["si"], "strength": r["strength"]})
    elif case["kind"] == "hamiltonian":
        state["rho"] = np.stack([v for _ in range(2) for v in _amplitudes(prob, rng)])
    else:
        state["xy"] = _amplitudes(prob, rng)
        state["h"] = np.stack([v for _ in range(2) for v in _amplitudes(prob, rng)])
    return state


def run(state):
    """The outputs of a solve are its strengths, iteration counts and, where
    asked for, amplitudes and cross-terms.  The last residual, which the call
    returns too, is what is left below the tolerance when two equal vectors are
    subtracted: no figure of it is determined by the inputs."""
    case, eng = state["case"], state["engine"]
    if case["kind"] == "hamiltonian":
        return {"h": eng.calc_hamiltonian(state["rho"])}
    if case["kind"] == "transforms":
        return {"sp": eng.qp2sp(*state["xy"]), "qp": eng.sp2qp(state["h"])}
    r = eng.solve(state["omega"], max_iter=300, eps=1e-7, broyden_history=50, precision=PRECISIONS[case["precision"]],
                  want_x=case["want_x"], restart=state.get("stored"))
    return {k: r[k] for k in ("strength", "iterations", "x", "crossterms") if k in r}


def work(case):
    """Bytes: per iteration the amplitudes of a point read and written, and the
    Broyden vectors it has by then read once.  Floating-point operations: the
    block transforms, and the densities and the projection contracted first
    along z and then along r (the basis functions are products of the two)."""
    prob = _prob(case)
    b, f = prob.basis, prob.f_struct
    db, nxy = np.asarray(b.db, dtype=np.float64), float(prob.nxy)
    transforms = 16.0 * sum(2 * db[i] * db[i] * db[j] + 2 * db[i] * db[j] * db[j] for i, j, _ in f.pairs())
    radial = [set(zip(b.nr[s:s + d], b.nl[s:s + d], b.ns[s:s + d])) for s, d in zip(b.isstart, b.db)]
    nrad = float(sum(len(radial[i]) * len(radial[j]) for i, j, _ in f.pairs()))
    grid = 2.0 * (16.0 * case["ngh"] * nxy + 44.0 * case["ngh"] * case["ngl"] * nrad)
    vec = 32.0 * nxy
    if case["kind"] == "hamiltonian":
        return {"bytes": 128.0 * nxy, "flops": 2.0 * grid}
    if case["kind"] == "transforms":
        return {"bytes": 192.0 * nxy, "flops": 2.0 * transforms}
    its = ITERATIONS * case["npts"]
    return {"bytes": its * vec * (4.0 + ITERATIONS / 2.0), "flops": its * 2.0 * (transforms + grid)}


# ---- the same in plain numpy -------------------------------------------------
def _maps(prob):
    """Column block of each row block: X, Y and the four density quadrants."""
    nb = prob.basis.nb
    tr = np.concatenate([np.arange(nb // 2, nb), np.arange(nb // 2)])
    f = np.asarray(prob.f_struct.ir2c)

    def inv(m):
        out = -np.ones(nb, dtype=np.int64)
        for i, j in enumerate(m):
            if j >= 0:
                out[j] = i
        return out
    x = np.where(f >= 0, tr[f], -1)
    y = f[tr]
    s22 = np.where(y >= 0, tr[y], -1)
    return f, x, y, [f, inv(x), inv(y), inv(s22)]


def _blocks(prob, m, re, im=None):
    """Stored elements -> {(row block, column block): matrix}."""
    db, out, at = prob.basis.db, {}, 0
    for i, j in enumerate(m):
        if j >= 0:
            n = int(db[i] * db[j])
            v = re[at:at + n] if im is None else re[at:at + n] + 1j * im[at:at + n]
            out[i, int(j)] = v.reshape(db[i], db[j], order="F")
            at += n
    return out


def _elements(blocks, m, n):
    out, at = np.zeros(n, dtype=np.complex128), 0
    for i, j in enumerate(m):
        if j >= 0:
            v = blocks[i, int(j)].ravel(order="F")
            out[at:at + v.size] = v
            at += v.size
    return out


def _mul(*fs):
    out = fs[0]
    for g in fs[1:]:
        rows = {}
        for (k, j), v in g.items():
            rows.setdefault(k, []).append((j, v))
        new = {}
        for (i, k), u in out.items():
            for j, v in rows.get(k, ()):
                new[i, j] = new[i, j] + u @ v if (i, j) in new else u @ v
        out = new
    return out


def _t(a):
    return {(j, i): v.T for (i, j), v in a.items()}


def _sum(*terms):
    out = {}
    for s, a in terms:
        for k, v in a.items():
            out[k] = out[k] + s * v if k in out else s * v
    return out


def _bogoliubov(prob):
    b = prob.basis
    nb = b.nb
    tr = np.concatenate([np.arange(nb // 2, nb), np.arange(nb // 2)])
    same = np.arange(nb)
    return [_blocks(prob, m, v) for m, v in ((same, b.Up), (tr, b.Vp), (same, b.Un), (tr, b.Vn))]


def _exact_transforms(prob, xy, h):
    n = prob.nxy
    f, x, y, dens = _maps(prob)
    Up, Vp, Un, Vn = _bogoliubov(prob)
    X, Y = _blocks(prob, x, xy[0], xy[1]), _blocks(prob, y, xy[2], xy[3])
    # W_p [[0, X], [-Y, 0]] W_n^T with W = [[U, V], [V, U]]
    s11 = _sum((1, _mul(Up, X, _t(Vn))), (-1, _mul(Vp, Y, _t(Un))))
    s12 = _sum((1, _mul(Up, X, _t(Un))), (-1, _mul(Vp, Y, _t(Vn))))
    s21 = _sum((1, _mul(Vp, X, _t(Vn))), (-1, _mul(Up, Y, _t(Un))))
    s22 = _sum((1, _mul(Vp, X, _t(Un))), (-1, _mul(Up, Y, _t(Vn))))
    quad = [s11, _sum((-1, _t(s12))), {k: v.conj() for k, v in _t(s21).items()}, _sum((-1, _t(s22)))]
    sp = []
    for q, m in zip(quad, dens):
        e = _elements(q, m, n)
        sp += [e.real, e.imag]
    # W_p^T [[h, D+], [-conj(D-), -h_np^T]] W_n
    h11, h12, hnp, dm = (_blocks(prob, m, h[2 * k], h[2 * k + 1]) for k, m in enumerate((f, x, f, y)))
    h21 = {k: -v.conj() for k, v in dm.items()}
    h22 = _sum((-1, _t(hnp)))
    q12 = _sum((1, _mul(_t(Up), h11, Vn)), (1, _mul(_t(Vp), h21, Vn)), (1, _mul(_t(Up), h12, Un)),
               (1, _mul(_t(Vp), h22, Un)))
    q21 = _sum((-1, _mul(_t(Vp), h11, Un)), (-1, _mul(_t(Up), h21, Un)), (-1, _mul(_t(Vp), h12, Vn)),
               (-1, _mul(_t(Up), h22, Vn)))
    h20, h02 = _elements(q12, x, n), _elements(q21, y, n)
    return {"sp": np.stack(sp), "qp": [h20.real, h20.imag, h02.real, h02.imag]}


def _products(prob, psi, blocks, only=None):
    """P[sa, sb][x, y](r) = sum_ab psi_x(r, a) rho(a, b) psi_y(r, b) over the
    rows of spin sa and the columns of spin sb (0 up, 1 down)."""
    b, g = prob.basis, prob.basis.nghl
    tabs = (0, 1, 2, 3) if only is None else only
    P = np.zeros((2, 2, 4, 4, g), dtype=np.complex128)
    for (i, j), rho in blocks.items():
        ri, rj, ui, uj = b.isstart[i], b.isstart[j], b.num_spin_up[i], b.num_spin_up[j]
        rows, cols = (slice(0, ui), slice(ui, b.db[i])), (slice(0, uj), slice(uj, b.db[j]))
        for x in tabs:
            A, full = psi[x][:, ri:ri + b.db[i]], psi
            for sa in (0, 1):
                if rows[sa].stop == rows[sa].start:
                    continue
                a = A[:, rows[sa]]
                T = a @ rho.real[rows[sa]] + 1j * (a @ rho.imag[rows[sa]])
                for y in tabs:
                    B = full[y][:, rj:rj + b.db[j]]
                    for sb in (0, 1):
                        P[sa, sb, x, y] += np.einsum("rb,rb->r", T[:, cols[sb]], B[:, cols[sb]])
    return P


def _exact_hamiltonian(prob, args):
    b, c, n = prob.basis, prob.couplings, prob.nxy
    f, x, y, dens = _maps(prob)
    psi = [np.asarray(v) for v in (b.wf, b.wfdr, b.wfdp, b.wfdz, b.wfd2_all)]
    (cdrho, ctau, ctj0, ctj1, ctj2, crdj, cds, ct, cj, cgs, cf, csdj) = c.scalars()
    crho, cs, cpair, cspair = c.crho, c.cs, c.cpair, c.cspair
    w = b.grid.wdcori
    out = []
    for sec, (mr, mk, mo, md) in enumerate(((dens[0], dens[1], f, x), (dens[3], dens[2], f, y))):
        P = _products(prob, psi, _blocks(prob, mr, args[4 * sec], args[4 * sec + 1])) * w
        kap = _products(prob, psi, _blocks(prob, mk, args[4 * sec + 2], args[4 * sec + 3]), (0,))[:, :, 0, 0] * w
        uu, dd, du, ud = P[0, 0], P[1, 1], P[1, 0], P[0, 1]
        p, m = uu + dd, uu - dd                       # same spin: sum, and with the sign of the spin
        q, e = ud + du, ud - du                       # opposite: sum, and + for (up, down), - for (down, up)
        rho, sz = p[0, 0], m[0, 0]
        jp, tjpz = 0.5 * (p[0, 2] + p[2, 0]), 0.5 * (m[0, 2] + m[2, 0])
        tz = m[1, 1] + m[2, 2] + m[3, 3]
        jr, tjrz = 0.5j * (p[0, 1] - p[1, 0]), 0.5j * (m[0, 1] - m[1, 0])
        jz, tjzz = 0.5j * (p[0, 3] - p[3, 0]), 0.5j * (m[0, 3] - m[3, 0])
        sr, sp = q[0, 0], 1j * e[0, 0]
        tjpr, tjpp = 0.5 * (q[2, 0] + q[0, 2]), 0.5j * (e[2, 0] + e[0, 2])
        gs = m[0, 3] + m[3, 0] + e[0, 2] - e[2, 0] + q[0, 1] + q[1, 0]
        tr, tp = q[1, 1] + q[2, 2] + q[3, 3], 1j * (e[1, 1] + e[2, 2] + e[3, 3])
        tjrr, tjrp = 0.5j * (q[0, 1] - q[1, 0]), -0.5 * (e[0, 1] - e[1, 0])
        tjzr, tjzp = 0.5j * (q[0, 3] - q[3, 0]), -0.5 * (e[0, 3] - e[3, 0])
        tau = p[1, 1] + p[2, 2] + p[3, 3]
        fr = 0.5 * (m[1, 3] + m[3, 1]) + q[1, 1] + 0.5 * (e[1, 2] - e[2, 1])
        fp = 1j * (0.5 * (m[2, 3] - m[3, 2]) + e[2, 2] + 0.5 * (q[2, 1] - q[1, 2]))
        fz = m[3, 3] + 0.5 * (q[3, 1] + q[1, 3] + e[3, 2] - e[2, 3])
        # pairing: kap[sa, sb]; columns of spin up count +, down -
        rb = 2.0 * (kap[0, 1] - kap[1, 0])
        sbz = 2.0 * (kap[0, 1] + kap[1, 0])
        sbr = 2.0 * (kap[1, 1] - kap[0, 0])
        sbp = -2.0j * (kap[0, 0] + kap[1, 1])
        c0 = ctj0 * (tjrr + tjpp + tjzz)
        c1a, c1b = ctj1 * (tjzr - tjrz), ctj1 * (tjpz - tjzp)
        c2a, c2b = ctj2 * (tjrz + tjzr), ctj2 * (tjpz + tjzp)
        mf = {}
        for sg, k in ((1.0, (0, 0)), (-1.0, (1, 1))):
            M = mf[k] = {}
            M[0, 0] = 2 * crho * rho + ctau * tau + sg * (2 * cs * sz + ct * tz + cf * fz)
            u, v = -crdj * (tjpz - tjzp) - sg * csdj * jp, 1j * (sg * (c1a - 0.5 * c2a) - cj * jr)
            M[0, 1], M[1, 0] = u + v, u - v
            u, v = cj * jp + sg * (c1b + 0.5 * c2b), 1j * (sg * csdj * jr - crdj * (tjzr - tjrz))
            M[0, 2], M[2, 0] = u + v, u - v
            u = -crdj * (tjrp - tjpr) + 2 * sg * cgs * gs
            v = -1j * (sg * (c0 - ctj2 / 3 * (tjrr + tjpp - 2 * tjzz)) + cj * jz)
            M[0, 3], M[3, 0] = u + v, u - v
            M[0, 4] = M[4, 0] = 2 * cdrho * rho + 2 * sg * cds * sz
            M[1, 2] = M[2, 1] = csdj * sz + sg * crdj * rho
            M[1, 3], M[3, 1] = 0.5 * sg * cf * sr + 1j * csdj * sp, 0.5 * sg * cf * sr - 1j * csdj * sp
            M[2, 3], M[3, 2] = -csdj * sr - 0.5j * sg * cf * sp, -csdj * sr + 0.5j * sg * cf * sp
            M[1, 1] = M[2, 2] = (4 * cdrho + ctau) * rho + sg * (4 * cds + ct) * sz
            M[3, 3] = M[1, 1] + sg * cf * sz
        a2, a3, a4 = -ctj1 * (tjrp - tjpr), -1j * c0, -0.5 * ctj2 * (tjrp + tjpr)
        a5, a6 = 1j * ctj2 / 3 * (tjpp + tjzz - 2 * tjrr), 1j * ctj2 / 3 * (tjrr + tjzz - 2 * tjpp)
        for ep, k in ((1.0, (0, 1)), (-1.0, (1, 0))):
            M = mf[k] = {}
            M[0, 0] = 2 * cs * sr + ct * tr + cf * fr - 1j * ep * (2 * cs * sp + ct * tp + cf * fp)
            g, iz = 2 * cgs * gs, 1j * csdj * jz
            u, v = g - ep * iz, ep * a2 + a3 + ep * a4 + a5
            M[0, 1], M[1, 0] = u + v, u - v
            u, v = a2 + ep * a3 - a4 + ep * a6, ep * g - iz
            M[0, 2], M[2, 0] = u + v, u - v
            u, v = csdj * (jp + 1j * ep * jr), -1j * (c1a + 0.5 * c2a) + ep * (c1b - 0.5 * c2b)
            M[0, 3], M[3, 0] = u + v, u - v
            M[0, 4] = M[4, 0] = 2 * cds * (sr - 1j * ep * sp)
            M[1, 2] = 0.5 * cf * (1j * sp + ep * sr)
            M[2, 1] = -M[1, 2]
            M[1, 3], M[3, 1] = 0.5 * cf * sz + ep * crdj * rho, 0.5 * cf * sz - ep * crdj * rho
            M[2, 3], M[3, 2] = -0.5 * ep * cf * sz - crdj * rho, 0.5 * ep * cf * sz - crdj * rho
            M[3, 3] = (ct + 4 * cds) * (sr - 1j * ep * sp)
            M[1, 1], M[2, 2] = M[3, 3] + cf * sr, M[3, 3] - 1j * ep * cf * sp
        pair = {(0, 0): cspair * (sbr - 1j * sbp), (1, 0): -cpair * rb - cspair * sbz,
                (0, 1): cpair * rb - cspair * sbz, (1, 1): cspair * (-sbr - 1j * sbp)}
        for mm, fields in ((mo, mf), (md, {k: {(0, 0): v} for k, v in pair.items()})):
            blocks = {}
            for i, j in enumerate(mm):
                if j < 0:
                    continue
                ri, rj, ui, uj = b.isstart[i], b.isstart[j], b.num_spin_up[i], b.num_spin_up[j]
                rows, cols = (slice(0, ui), slice(ui, b.db[i])), (slice(0, uj), slice(uj, b.db[j]))
                H = np.zeros((b.db[i], b.db[j]), dtype=np.complex128)
                for (sa, sb), M in fields.items():
                    if rows[sa].stop == rows[sa].start or cols[sb].stop == cols[sb].start:
                        continue
                    for z in sorted({k[0] for k in M}):
                        B = sum(v[:, None] * psi[k[1]][:, rj:rj + b.db[j]][:, cols[sb]] for k, v in M.items()
                                if k[0] == z)
                        A = psi[z][:, ri:ri + b.db[i]][:, rows[sa]].T
                        H[rows[sa], cols[sb]] += 2.0 * (A @ B.real + 1j * (A @ B.imag))
                blocks[i, int(j)] = H
            e = _elements(blocks, mm, n)
            out += [e.real, e.imag]
    return {"h": np.stack(out)}


def exact(case, seed):
    """Plain numpy for the linear calls.  A converged solve has no such value:
    where between the tolerance and zero its residual ends, and with it the last
    figures of the strength, is up to the iteration."""
    if case["kind"] not in ("hamiltonian", "transforms"):
        return None
    prob = _prob(case)
    if case["kind"] == "hamiltonian" and prob.nxy * float(prob.basis.nghl) > 2.0e8:
        return None          # above 20 seconds on the host
    rng = np.random.default_rng([seed, case["nsh"], case["npts"]])
    if case["kind"] == "hamiltonian":
        return _exact_hamiltonian(prob, np.stack([v for _ in range(2) for v in _amplitudes(prob, rng)]))
    xy = _amplitudes(prob, rng)
    return _exact_transforms(prob, xy, np.stack([v for _ in range(2) for v in _amplitudes(prob, rng)]))
