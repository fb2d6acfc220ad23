"""The calls by which this framework's speed is judged: core-level BSE problems, from the
smallest meshes of the tests to the L2,3 workload of the benchmark, through the public
entry points of ocean_amd.core.

A case is one call as a program makes it on a problem that it has loaded: the Lanczos
recursion with its spectrum (the main use), several polarisations or several problems at
once, GMRES at a few energies, the bi-Lanczos recursion, the OBF form, one action on host
planes, and the gradient of a spectral misfit.  Inputs have the distributions of
ocean_amd.synth; the Bloch functions are orthonormal over x at each k and drawn on the GPU.
Results of the mixed form are kept in single precision, as they carry about seven digits.
"""
import math

import numpy as np
import torch

from ocean_amd import core, setup_host, synth

EV = core.EV2HARTREE
EL, EH, GAM, NE = -5.0, 40.0, 0.5, 2000   # the spectrum's window and broadening (eV), points
DENSE = 4200                               # the largest operator that exact() forms whole


def _case(name, kind, nb, k, x, **more):
    c = {"name": name, "kind": kind, "nb": nb, "k1": k[0], "k2": k[1], "k3": k[2],
         "x1": x[0], "x2": x[1], "x3": x[2], "lc": 0, "nspn": 1, "mixed": False, "nrhs": 1, "niter": 40}
    c.update(more)
    return c


def listed():
    return [
        # the drop-in call of a host program that keeps its vectors: one action, host planes
        # in and out, on a small ragged mesh with two spins
        _case("action_small", "action", 18, (3, 4, 5), (5, 6, 7), nspn=2),
        # the smallest solve of the tests and the benchmark's smallest workload
        _case("haydock_k16", "haydock", 16, (4, 4, 4), (6, 6, 6)),
        # the drop-in timing workload, K edge
        _case("haydock_k64", "haydock", 64, (8, 8, 8), (8, 8, 8)),
        _case("haydock_k64_mixed", "haydock", 64, (8, 8, 8), (8, 8, 8), mixed=True),
        # L2,3 edge (twelve alphas, spin-orbit), 128 bands, the largest problem
        _case("haydock_l23", "haydock", 128, (8, 8, 8), (10, 10, 10), lc=1),
        _case("haydock_l23_mixed", "haydock", 128, (8, 8, 8), (10, 10, 10), lc=1, mixed=True),
        # three polarisations of one site sharing its Hamiltonian
        _case("multi3_k64", "multi", 64, (8, 8, 8), (8, 8, 8), nrhs=3),
        # an uneven batch of K and L2,3 edges, mixed precision, as the benchmark's batch
        _case("batch_mixed", "batch", 64, (8, 8, 8), (8, 8, 8), mixed=True, members=6, pick=5, niter=24),
        # GMRES over a few energies at the timing workload, and on an odd mesh with solutions
        _case("gmres_k64", "gmres", 64, (8, 8, 8), (8, 8, 8), energies=4, depth=100, with_x=False),
        _case("gmres_odd", "gmres", 13, (3, 4, 5), (5, 6, 7), energies=6, depth=80, with_x=True),
        # the orbital-basis form of the long-range term
        _case("obf_k64", "obf", 64, (8, 8, 8), (8, 8, 8), num_obf=128),
        # forward and adjoint solves and the derivative with respect to the W table
        _case("gradient_k16", "gradient", 16, (4, 4, 4), (6, 6, 6), energies=4, depth=80),
    ]


def draw(rng):
    kind = rng.choices(["haydock", "multi", "batch", "gmres", "obf", "abc", "action", "gradient"],
                       [8, 2, 2, 2, 1, 1, 1, 1])[0]
    small = kind in ("gmres", "gradient", "abc", "action")
    while True:
        if rng.random() < 0.4:
            k = (rng.randint(2, 8),) * 3
        else:
            k = tuple(rng.randint(2, 8) for _ in range(3))
        x = tuple(rng.randint(4, 8 if small else 10) for _ in range(3))
        nk, nx = k[0] * k[1] * k[2], x[0] * x[1] * x[2]
        nb = int(round(math.exp(rng.uniform(math.log(8), math.log(128)))))
        lc = 1 if rng.random() < 0.35 else 0
        nspn = 2 if rng.random() < 0.2 else 1
        if kind in ("multi", "obf"):
            nspn = 1
        if kind in ("multi", "gradient"):
            lc = 0
        most = 3_000_000 if kind == "gradient" else 17_000_000 if small else 40_000_000
        if nb <= nx and 50_000 <= nb * nk * nx * nspn * (3 if lc else 1) <= most:
            break
    mixed = kind in ("haydock", "multi", "batch") and rng.random() < 0.4
    c = _case("", kind, nb, k, x, lc=lc, nspn=nspn, mixed=mixed, niter=rng.randint(16, 40))
    del c["name"]
    if kind == "multi":
        c["nrhs"] = rng.choice([3, 6])
    elif kind == "batch":
        c.update(members=rng.randint(3, 6), pick=rng.randint(0, 99), nspn=1, lc=0, niter=rng.randint(12, 24))
    elif kind == "gmres":
        c.update(energies=rng.randint(2, 4), depth=rng.randint(80, 100), with_x=rng.random() < 0.5)
    elif kind == "gradient":
        c.update(energies=rng.randint(2, 4), depth=rng.randint(80, 100), nspn=1)
    elif kind == "obf":
        c["num_obf"] = rng.randint(min(nb, nx), min(nx, 2 * nb + 8))
    return c


def _members(case):
    """The problems of a batch: its own sizes first, then members of the benchmark's batch."""
    if case["kind"] != "batch":
        return [case]
    rng = np.random.default_rng(case["pick"])
    pool = [m for m in synth.batch_members(96) if m["kmesh"][0] <= 6 or m["nb"] <= 64]
    out = [case]
    for i in rng.permutation(len(pool))[:case["members"] - 1]:
        m = pool[int(i)]
        out.append(dict(case, nb=m["nb"], lc=m["lc"], k1=m["kmesh"][0], k2=m["kmesh"][1], k3=m["kmesh"][2],
                        x1=m["xmesh"][0], x2=m["xmesh"][1], x3=m["xmesh"][2]))
    return out


def _sizes(case):
    nk, nx = case["k1"] * case["k2"] * case["k3"], case["x1"] * case["x2"] * case["x3"]
    return case["nb"], nk, nx, 4 * (2 * case["lc"] + 1), case["nspn"]


def _orthonormal(gen, *shape):
    """Gaussian columns made orthonormal over the next-to-last axis (Newton-Schulz)."""
    z = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.complex128) / math.sqrt(shape[-2])
    eye = torch.eye(shape[-1], device="cuda", dtype=torch.complex128)
    z = z / (1.0 + math.sqrt(shape[-1] / shape[-2]))
    for _ in range(9):
        z = torch.matmul(z, 1.5 * eye - 0.5 * torch.matmul(z.mH.contiguous(), z))
    return z


def _inputs(case, seed):
    """One problem's inputs: ocean_amd.synth's, with the Bloch functions u (s, k, x, n) on the GPU."""
    nb, nk, nx, na, ns = _sizes(case)
    inp = synth.make_inputs(nb, (case["k1"], case["k2"], case["k3"]), (case["x1"], case["x2"], case["x3"]),
                            lc=case["lc"], nspn=ns, seed=seed, xi_eV=10.0 / 1.5 if case["lc"] else 0.0, with_u=False)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    obf = u = None
    if case["kind"] == "obf":
        obf = synth.make_obf(inp, case["num_obf"], seed=seed)
    else:
        u = _orthonormal(gen, ns, nk, nx, nb)
    psis = [inp.psi0]
    rng = np.random.default_rng(seed + 1)
    for _ in range(case["nrhs"] - 1):
        z = rng.standard_normal(inp.psi0.shape) + 1j * rng.standard_normal(inp.psi0.shape)
        psis.append(setup_host.normalise_psi0(np.asfortranarray(z), nk, inp.celvol)[0])
    return inp, u, obf, psis


def _handle(case, inp, u, obf):
    g = core.OceanGPU.from_inputs(inp, precision=core.MIXED if case["mixed"] else core.FP64, nrhs=case["nrhs"])
    if obf is not None:
        g.load_w(obf.W)
        g.load_obf(obf.obf, obf.obf2u, obf.xoff)
    else:
        planes = u.permute(0, 2, 1, 3)  # (s, x, k, n): the host program's order, bands fastest
        re, im = planes.real.contiguous(), planes.imag.contiguous()
        torch.cuda.synchronize()
        g.load_bloch_dev(re.data_ptr(), im.data_ptr())
    return g


def _energies(case):
    return np.linspace(-2.0, 25.0, case["energies"])


def _rdist(inp):
    return setup_host.w_geometry(inp.avec, inp.kmesh, inp.xmesh, inp.tau, inp.xshift)[0]


def _target(case, seed):
    rng = np.random.default_rng(seed + 2)
    return 0.05 * rng.uniform(0.5, 1.5, case["energies"])


def prepare(case, seed):
    s = {"case": case, "g": [], "psi": [], "kpref": []}
    for i, m in enumerate(_members(case)):
        inp, u, obf, psis = _inputs(m, seed + 1000 * i)
        g = _handle(m, inp, u, obf)
        if case["kind"] == "gradient":
            g.build_w(_rdist(inp), inp.rtab, inp.ptab, inp.epsilon0, inp.inter_scale)
            s["target"] = _target(case, seed)
        s["g"].append(g)
        s["psi"].append(np.stack(psis) if case["nrhs"] > 1 else psis[0])
        s["kpref"].append(inp.kpref)
    if case["kind"] == "batch":
        s["batch"] = core.OceanBatch(s["g"])
    return s


def _kept(case, v):
    """What the program keeps of a recursion: single precision where the form is the mixed one."""
    return {k: np.asarray(a, np.float32) if case["mixed"] else a for k, a in v.items()}


def _spectrum(a, b, n, kpref):
    return core.spectrum(a, b, n, kpref, GAM * EV, EL * EV, EH * EV, NE, literal_cmplx=False)


def run(s):
    case, g, psi, kpref, n = s["case"], s["g"][0], s["psi"][0], s["kpref"][0], s["case"]["niter"]
    kind = case["kind"]
    if kind == "action":
        return {"forward": g.xact(psi), "backward": g.xact(psi, backwards=True)}
    if kind in ("haydock", "obf"):
        a, b, _ = g.haydock(psi, n)
        return _kept(case, {"a": a, "b": b, "spectrum": _spectrum(a, b, n, kpref)})
    if kind == "multi":
        a, b, _ = g.haydock_multi(psi, n)
        return _kept(case, {"a": a, "b": b,
                            "spectra": np.stack([_spectrum(a[r], b[r], n, kpref) for r in range(case["nrhs"])])})
    if kind == "batch":
        got, _ = s["batch"].haydock(s["psi"], n)
        return [_kept(case, {"a": a, "b": b, "spectrum": _spectrum(a, b, n, kp)})
                for (a, b, _), kp in zip(got, s["kpref"])]
    if kind == "abc":
        co = g.haydock_abc(psi, n)
        return {"a": co[0] + 1j * co[1], "b": co[2] + 1j * co[3], "c": co[4] + 1j * co[5],
                "spectrum": core.spectrum_abc(*co, n, kpref, GAM * EV, EL * EV, EH * EV, NE, literal_cmplx=False)}
    if kind == "gmres":
        got = g.gmres(psi, _energies(case), GAM, 13.605, 1e-14, case["depth"], kpref=kpref, return_x=case["with_x"])
        return {"rows": got[0], "x": got[1]} if case["with_x"] else {"rows": got}
    if kind == "gradient":
        r = g.spectral_grad(psi, _energies(case), GAM, 13.605, 1e-16, case["depth"], s["target"], kpref=kpref)
        return {k: r[k] for k in ("loss", "sigma", "g_ptab", "g_scale", "g_gamma_eV", "g_scissor_eV")}
    raise ValueError(kind)


def work(case):
    """u is read once per action (what every form needs), the vectors once per step."""
    by = fl = 0.0
    for m in _members(case):
        nb, nk, nx, na, ns = _sizes(m)
        na *= m["nrhs"]
        P, N, el = 16, nb * nk * na, 4 if m["mixed"] else 8
        if m["kind"] == "obf":
            no = m["num_obf"]
            one_b = 16.0 * nb * nk * no + 16.0 * no * nx + 8.0 * nk * nx + 56.0 * N
            one_f = 16.0 * na * nk * (nb * no + no * nx)
        else:
            one_b = 2.0 * el * nb * nk * nx * ns + el * nk * nx + 16.0 * nb * nk * P * ns + 56.0 * N
            one_f = 16.0 * nb * nk * nx * na
        fft = 10.0 * nk * math.log2(max(nk, 2)) * nx * na
        acts = {"haydock": m["niter"], "multi": m["niter"], "batch": m["niter"], "obf": m["niter"], "abc": 2 * m["niter"],
                "action": 2, "gmres": 40 * m.get("energies", 0), "gradient": 80 * m.get("energies", 0)}[m["kind"]]
        by += acts * (one_b + 16.0 * N)
        fl += acts * (one_f + fft + 16.0 * P * N)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------------------
# The same results in 64-bit torch, from the formulas
# ---------------------------------------------------------------------------
def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


class _Operator:
    """H of one right-hand side on arrays (k, n, a)."""

    def __init__(self, case, inp, u, obf):
        nb, nk, nx, na, ns = _sizes(case)
        self.km, self.nk, self.na, self.ns = (case["k1"], case["k2"], case["k3"]), nk, na, ns
        self.u = u
        self.W = _t(np.asarray(obf.W if obf is not None else inp.W)).to(torch.complex128)  # (k, x)
        self.E = _t(np.transpose(inp.energy, (1, 0, 2)))
        self.m = inp.mult
        self.obf = None
        self.with_mult = obf is None
        if obf is not None:
            km, xm = np.array(self.km), np.array([case["x1"], case["x2"], case["x3"]])
            q = np.stack([v.ravel() for v in np.meshgrid(*[np.arange(n) for n in km], indexing="ij")], axis=1)
            ph = 2 * np.pi * (q / (km * xm)) @ obf.xoff.T.astype(np.float64)  # (k, x)
            self.obf = (_t(np.transpose(obf.obf2u, (2, 0, 1))), _t(obf.obf), _t(np.exp(1j * ph)))
        # projectors c (s, k, n, p) and K over (a, p): -mpm on the diagonal of alpha, plus the exchange blocks
        m, cols, pl = self.m, [], []
        for li, l in enumerate(range(m.lmin, m.lmax + 1)):
            for mm in range(-l, l + 1):
                cols.append(np.transpose(m.c[:, :, 0, mm + m.lmax, li, :], (2, 1, 0)))
                pl.append(li)
        self.c = _t(np.stack(cols, axis=-1))
        P = len(pl)
        K = np.zeros((na, P, na, P), np.complex128)
        at = 0
        for li, l in enumerate(range(m.lmin, m.lmax + 1)):
            w = 2 * l + 1
            X = np.asarray(m.X[li]).T.reshape(na, w, na, w)  # the action takes mh(jj, ii)
            K[:, at:at + w, :, at:at + w] += X
            for a in range(na):
                for j in range(w):
                    K[a, at + j, a, at + j] -= m.mpm[0, 0, li]
            at += w
        self.K = _t(K.reshape(na * P, na * P))
        self.mul = inp.inter_scale / (nk * inp.celvol)
        self.S = _t(m.somelr + 1j * m.someli)
        self.spin = [slice(None)] if ns == 1 else [slice(0, None, 2), slice(1, None, 2)]

    def field(self, v):
        """F_+ (U v) as (a, k, x), with the transform over k unnormalised."""
        out = torch.empty(self.na, *self.km, self.W.shape[1], device="cuda", dtype=torch.complex128)
        for s, sl in enumerate(self.spin):
            phi = torch.matmul(self.u[s], v[:, :, sl].contiguous())          # (k, x, a)
            p = phi.permute(2, 0, 1).reshape(-1, *self.km, phi.shape[1])
            out[sl] = torch.fft.ifftn(p, dim=(1, 2, 3), norm="forward")
        return out.reshape(self.na, self.nk, -1)

    def _smooth(self, phi):
        """F_- W F_+ of (k, x, a), unnormalised."""
        p = phi.permute(2, 0, 1).reshape(phi.shape[2], *self.km, phi.shape[1])
        p = torch.fft.ifftn(p, dim=(1, 2, 3), norm="forward") * self.W.reshape(*self.km, -1)
        return torch.fft.fftn(p, dim=(1, 2, 3)).reshape(phi.shape[2], self.nk, -1).permute(1, 2, 0).contiguous()

    def long_range(self, v):
        if self.obf is not None:
            c2, f, ph = self.obf
            phi = torch.matmul(f.T.contiguous(), torch.matmul(c2.transpose(1, 2).contiguous(), v)) * ph[:, :, None]
            y = self._smooth(phi) * ph.conj()[:, :, None]
            return torch.matmul(c2.conj().resolve_conj().contiguous(), torch.matmul(f.conj().resolve_conj().contiguous(), y))
        out = torch.empty_like(v)
        for s, sl in enumerate(self.spin):
            y = self._smooth(torch.matmul(self.u[s], v[:, :, sl].contiguous())) / self.nk
            out[:, :, sl] = -torch.matmul(self.u[s].mH.resolve_conj().contiguous(), y)
        return out

    def multiplet(self, v):
        amp = torch.zeros(self.na, self.c.shape[-1], device="cuda", dtype=torch.complex128)
        for s, sl in enumerate(self.spin):
            amp[sl] = torch.matmul(self.c[s].reshape(-1, self.c.shape[-1]).T.contiguous(),
                                   v[:, :, sl].reshape(-1, v[:, :, sl].shape[2]).contiguous()).T
        h = self.mul * (self.K @ amp.reshape(-1)).reshape(self.na, -1)
        out = torch.empty_like(v)
        for s, sl in enumerate(self.spin):
            out[:, :, sl] = torch.matmul(self.c[s].conj().resolve_conj().contiguous(), h[sl].T.contiguous())
        return out

    def interaction(self, v):
        return self.long_range(v) + (self.multiplet(v) if self.with_mult else 0)

    def __call__(self, v, back=False):
        out = (self.E.conj() if back else self.E) * v + self.interaction(v)
        if self.m.have_spin_orbit:
            out = out + torch.matmul(v, (self.S.conj() if back else self.S).T.contiguous())
        return out

    def dense(self, n):
        eye = torch.eye(self.nk * n * self.na, device="cuda", dtype=torch.complex128)
        cols = [self(e.reshape(self.nk, n, self.na)).reshape(-1) for e in eye]
        return torch.stack(cols, dim=1)


def _vec(psi):
    return _t(np.transpose(psi, (1, 0, 2)))


def _back(v):
    return np.transpose(v.cpu().numpy(), (1, 0, 2))


def _fraction(a, b, c, n, kpref):
    """The continued fraction with its square-root terminator, rows as core.spectrum's."""
    ie = np.arange(NE + 1)
    e = EL * EV + (EH - EL) * EV * (2.0 * ie) / (2.0 * NE)
    g = GAM * EV
    ct = e - a[n - 1].real + 1j * (g + a[n - 1].imag)
    disc = np.sqrt(ct * ct - 4.0 * b[n] * c[n] + 0j)
    d = np.where(disc.imag > 0.0, 0.5 * (ct + disc), 0.5 * (ct - disc))
    for j in range(n - 1, -1, -1):
        d = (e - a[j].real + 1j * (g + a[j].imag)) - b[j + 1] * c[j + 1] / d
    d = d.real + 1j * np.abs(d.imag)
    den = np.abs(d) ** 2
    sp, kk = kpref * d.imag / den, kpref * d.real / den
    return np.stack([core.HARTREE2EV * e, sp, sp, kk, kk], axis=1)


def _lanczos(H, psi, n):
    a, b = np.zeros(n + 1), np.zeros(n + 1)
    v, old = _vec(psi), 0.0
    for i in range(1, n + 1):
        h = H(v) - b[i - 1] * old
        a[i - 1] = float(torch.vdot(v.reshape(-1), h.reshape(-1)).real)
        h = h - a[i - 1] * v
        b[i] = float(torch.linalg.norm(h.reshape(-1)))
        old, v = v, h / b[i]
    return a, b


def _bilanczos(H, psi, n):
    """As OCEAN2 runs it: h and its back vector, c = sqrt(<bh|h>), b = conj(<bh|h> / c)."""
    a, b, c = (np.zeros(n + 1, complex) for _ in range(3))
    v = w = _vec(psi)
    vo = wo = 0.0
    for i in range(1, n + 1):
        h, k = H(v), H(w, back=True)
        a[i - 1] = complex(torch.vdot(w.reshape(-1), h.reshape(-1)))
        h = h - b[i - 1] * vo - a[i - 1] * v
        k = k - np.conj(c[i - 1]) * wo - np.conj(a[i - 1]) * w
        r = complex(torch.vdot(k.reshape(-1), h.reshape(-1)))
        c[i] = np.sqrt(r)
        b[i] = np.conj(r / c[i])
        vo, wo, v, w = v, w, h / c[i], k / np.conj(b[i])
    return a, b, c


def _exact_gradient(case, seed, inp, H, psi):
    """Loss, spectrum and derivatives from dense solves (E + i Gamma - H) x = b."""
    A = H.dense(case["nb"])
    bv = _vec(psi).reshape(-1)
    eye = torch.eye(bv.numel(), device="cuda", dtype=torch.complex128)
    sig, tgt = np.zeros(case["energies"]), _target(case, seed)
    Q = torch.zeros(H.W.shape, device="cuda", dtype=torch.float64)
    gG = gD = gS = 0.0
    for i, e in enumerate(_energies(case) * EV):
        M = (e + 1j * GAM * EV) * eye - A
        lu = torch.linalg.lu_factor(M)
        x = torch.linalg.lu_solve(*lu, bv[:, None])[:, 0]
        y = torch.linalg.solve(M.mH.resolve_conj().contiguous(), bv[:, None])[:, 0]
        sig[i] = -inp.kpref * float(torch.vdot(bv, x).imag)
        c = 2.0 * (sig[i] - tgt[i]) * inp.kpref
        yx = complex(torch.vdot(y, x))
        gG += c * yx.real
        gD -= c * yx.imag
        shape = (H.nk, case["nb"], H.na)
        gS -= c * complex(torch.vdot(y, H.interaction(x.reshape(shape)).reshape(-1))).imag / inp.inter_scale
        px, py = H.field(x.reshape(shape)), H.field(y.reshape(shape))
        Q += c / H.nk * (py.conj() * px).sum(0).imag
    # W(k, x) is linear in two knots of its table
    r, rt = _rdist(inp), np.asarray(inp.rtab)
    q, g = Q.cpu().numpy(), np.zeros(len(rt))
    j = np.clip(np.searchsorted(rt, r, side="left") - 1, 0, len(rt) - 2)
    t = (r - rt[j]) / (rt[j + 1] - rt[j])
    t = np.where(r < rt[0], 0.0, t)
    inside = (r <= rt[-1]) * inp.inter_scale
    np.add.at(g, j, q * (1.0 - t) * inside)
    np.add.at(g, j + 1, q * t * inside)
    return {"loss": float(((sig - tgt) ** 2).sum()), "sigma": sig, "g_ptab": g, "g_scale": gS, "g_gamma_eV": gG * EV,
            "g_scissor_eV": gD * EV}


def exact(case, seed):
    kind, n = case["kind"], case["niter"]
    nb, nk, nx, na, ns = _sizes(case)
    if kind in ("gmres", "gradient") and nb * nk * na > DENSE:
        return None
    out = []
    for i, m in enumerate(_members(case)):
        inp, u, obf, psis = _inputs(m, seed + 1000 * i)
        H = _Operator(m, inp, u, obf)
        if kind == "action":
            return {"forward": _back(H(_vec(psis[0]))), "backward": _back(H(_vec(psis[0]), back=True))}
        if kind == "gradient":
            return _exact_gradient(case, seed, inp, H, psis[0])
        if kind == "gmres":
            A, bv = H.dense(nb), _vec(psis[0]).reshape(-1)
            eye = torch.eye(bv.numel(), device="cuda", dtype=torch.complex128)
            xs = [torch.linalg.solve((e + 1j * GAM * EV) * eye - A, bv[:, None]).reshape(nk, nb, na)
                  for e in _energies(case) * EV]
            return {"rows": None, "x": np.stack([_back(x) for x in xs], axis=3)} if case["with_x"] else None
        if kind == "abc":
            a, b, c = _bilanczos(H, psis[0], n)
            return {"a": a, "b": b, "c": c, "spectrum": _fraction(a, b, c, n, inp.kpref)}
        got = []
        for p in psis:
            a, b = _lanczos(H, p, n)
            got.append((a, b, _fraction(a, b, b, n, inp.kpref)))
        if kind == "multi":
            return {k: np.stack([g[j] for g in got]) for j, k in enumerate(("a", "b", "spectra"))}
        out.append({"a": got[0][0], "b": got[0][1], "spectrum": got[0][2]})
    return out if kind == "batch" else out[0]
