"""The Haydock recursion at every thread budget of the adjoint, whose epilogue also sums
<h|psi>: workgroups of bands that do and do not divide a wave, budgets of one wave and up,
both adjoint forms, one and two spins, several right-hand sides and the OBF form.  FP64
against the oracle's recursion at the bar of the other recursion tests; the mixed form's
first coefficients within its H.psi bar (1e-5 of the largest element, so at most
1e-5 max|H psi| sqrt(N) in any product with a normalised vector)."""
import numpy as np
import pytest

import ocean_oracle as orc
from helpers import to_problem

pytestmark = pytest.mark.gpu

from ocean_amd import core, synth  # noqa: E402

N = 12
SPECS = {
    "nb5": dict(nb=5, kmesh=(2, 3, 2), xmesh=(3, 3, 2), seed=111),     # 60 of 64 threads
    "nb33": dict(nb=33, kmesh=(2, 2, 2), xmesh=(5, 3, 3), seed=112),   # 33 of 64, 99 of 128
    "nb64": dict(nb=64, kmesh=(2, 2, 1), xmesh=(4, 4, 5), seed=113),   # whole waves
    "nb100": dict(nb=100, kmesh=(2, 1, 2), xmesh=(5, 5, 5), seed=114),  # from a budget of 128
    "spin2": dict(nb=18, kmesh=(3, 2, 2), xmesh=(3, 3, 4), nspn=2, seed=115),
    "l23": dict(nb=13, kmesh=(2, 2, 3), xmesh=(3, 3, 3), lc=1, seed=116, xi_eV=3.0),
}


def _check(a, b, ref, what):
    ra, rb = ref
    assert np.max(np.abs(a[:N] - ra[:N]) / np.abs(ra[:N])) < 1e-10, what
    assert np.max(np.abs(b[1:N + 1] - rb[1:N + 1]) / np.abs(rb[1:N + 1])) < 1e-10, what


@pytest.mark.parametrize("name,adj", [(n, t) for n in SPECS for t in (64, 128, 256, 512) if t >= SPECS[n]["nb"]])
def test_haydock_at_adjoint_budget(name, adj):
    inp = synth.make_inputs(**SPECS[name])
    P = to_problem(inp)
    ra, rb, _, ierr = orc.haydock(P, inp.psi0, N)
    assert ierr == 0
    h = orc.xact(P, inp.psi0)
    bar = 1e-5 * np.abs(h).max() * np.sqrt(h.size)
    with core.OceanGPU.from_inputs(inp) as g:
        for form in (0, 1):
            g.set_tiles(256, adj, 0, form)
            g.set_precision(core.FP64)
            a, b, _ = g.haydock(inp.psi0, N)
            _check(a, b, (ra, rb), (name, adj, form))
            g.set_precision(core.MIXED)
            a, b, _ = g.haydock(inp.psi0, 1)
            assert abs(a[0] - ra[0]) < bar and abs(b[1] - rb[1]) < 2 * bar, (name, adj, form)


@pytest.mark.parametrize("adj", [64, 256])
def test_haydock_multi_at_adjoint_budget(adj):
    """Three right-hand sides on one spin (the vector-unit adjoint by choice) and on two."""
    for kw in (dict(nb=13, kmesh=(2, 2, 3), xmesh=(3, 3, 3), seed=117),
               dict(nb=33, kmesh=(2, 2, 1), xmesh=(4, 3, 3), nspn=2, seed=118)):
        inp = synth.make_inputs(**kw)
        P = to_problem(inp)
        rng = np.random.default_rng(8)
        psis = []
        for _ in range(3):
            z = rng.standard_normal(inp.psi0.shape) + 1j * rng.standard_normal(inp.psi0.shape)
            psis.append(np.asfortranarray(z / np.linalg.norm(z)))
        with core.OceanGPU.from_inputs(inp, nrhs=3) as g:
            g.set_tiles(256, adj, 0, 0)
            a, b, _ = g.haydock_multi(psis, N)
        for r, p in enumerate(psis):
            ra, rb, _, ierr = orc.haydock(P, p, N)
            assert ierr == 0
            _check(a[r], b[r], (ra, rb), (kw["nb"], adj, r))


@pytest.mark.parametrize("adj", [64, 256])
def test_haydock_obf_at_adjoint_budget(adj):
    inp = synth.make_inputs(nb=13, kmesh=(3, 4, 2), xmesh=(4, 3, 5), seed=119)
    ob = synth.make_obf(inp, 37, seed=120)
    phs = orc.obf_phase(inp.xmesh, inp.kmesh, inp.tau + inp.xshift / np.array(inp.xmesh, float))[0]
    P = to_problem(inp)
    P.W = ob.W
    ra, rb, _, ierr = orc.haydock(P, inp.psi0, N, act=lambda v: orc.xact_obf(P, v, ob.obf, ob.obf2u, phs))
    assert ierr == 0
    with core.OceanGPU.from_inputs(inp) as g:
        g.load_w(ob.W)
        g.load_obf(ob.obf, ob.obf2u, ob.xoff)
        g.set_tiles(256, adj, 0, -1)
        a, b, _ = g.haydock(inp.psi0, N)
    _check(a, b, (ra, rb), adj)


@pytest.mark.parametrize("kw,nrhs,n", [
    (dict(nb=3, kmesh=(1, 1, 1), xmesh=(3, 2, 1), seed=121), 1, 5),    # one partial; the Krylov space has 6 vectors
    (dict(nb=65, kmesh=(3, 5, 5), xmesh=(5, 14, 1), seed=122), 1, N),  # 38 partials
    (dict(nb=9, kmesh=(8, 8, 5), xmesh=(3, 3, 1), lc=1, lmax=4, seed=123, xi_eV=2.0), 2, N),
    (dict(nb=18, kmesh=(3, 4, 5), xmesh=(3, 3, 2), nspn=2, seed=124), 1, N)])
def test_haydock_without_the_long_range_term(kw, nrhs, n):
    """The multiplet term's own two kernels (no transform to ride on) and b finished on its
    own: 1 to 64 partials, 16 and 25 projectors, two spins, two right-hand sides."""
    inp = synth.make_inputs(**kw)
    P = to_problem(inp, long_range=False)
    rng = np.random.default_rng(9)
    psis = []
    for _ in range(nrhs):
        z = rng.standard_normal(inp.psi0.shape) + 1j * rng.standard_normal(inp.psi0.shape)
        psis.append(np.asfortranarray(z / np.linalg.norm(z)))
    with core.OceanGPU.from_inputs(inp, long_range=False, nrhs=nrhs) as g:
        a, b, _ = g.haydock_multi(psis, n)
    for r, p in enumerate(psis):
        ra, rb, _, ierr = orc.haydock(P, p, n)
        assert ierr == 0
        assert np.max(np.abs(a[r, :n] - ra[:n]) / np.abs(ra[:n])) < 1e-10
        assert np.max(np.abs(b[r, 1:n + 1] - rb[1:n + 1]) / np.abs(rb[1:n + 1])) < 1e-10
