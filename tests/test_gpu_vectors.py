"""Host vectors and workspaces: the interleaved entry points against the ones with planes,
vectors long enough to be staged in parts, and workspaces that other solves have used."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from ocean_amd import core, synth  # noqa: E402


def _planes_haydock(g, psi, niter):
    re, im = np.asfortranarray(psi.real), np.asfortranarray(psi.imag)
    a, b, ai = (np.zeros(niter + 1) for _ in range(3))
    done = C.c_int32()
    rc = core._lib().ocean_gpu_haydock(g.h, core._p(re), core._p(im), niter, core._p(a), core._p(b), core._p(ai),
                                       C.byref(done))
    assert rc == 0 and done.value == niter
    return a, b, ai


# 2 560 elements; 393 216, past the 262 144 from which a vector is staged in four parts
@pytest.mark.parametrize("nb,kmesh,xmesh,lc", [(10, (4, 4, 4), (3, 3, 2), 0), (64, (8, 8, 8), (4, 4, 4), 1)])
def test_interleaved_and_planes_agree(nb, kmesh, xmesh, lc):
    inp = synth.make_inputs(nb=nb, kmesh=kmesh, xmesh=xmesh, lc=lc, seed=95, xi_eV=3.0 if lc else 0.0)
    rng = np.random.default_rng(3)
    with core.OceanGPU.from_inputs(inp) as g:
        z = np.asfortranarray(rng.standard_normal(g.shape) + 1j * rng.standard_normal(g.shape))
        v = g.vec_new(z)
        assert np.array_equal(g.vec_get(v), z)
        want = _planes_haydock(g, inp.psi0, 3)
        for psi in (inp.psi0, np.ascontiguousarray(inp.psi0)):  # held in the library's order, and not
            for x, y in zip(g.haydock(psi, 3), want):
                assert np.array_equal(x, y)


def test_workspace_is_shared_by_the_solves():
    """Recursions before and after a GMRES solve on the same handle (its vectors take the
    same workspace) and another length of recursion give the same coefficients."""
    inp = synth.make_inputs(nb=9, kmesh=(3, 2, 4), xmesh=(3, 3, 3), lc=0, seed=96)
    with core.OceanGPU.from_inputs(inp) as g:
        first = g.haydock(inp.psi0, 12)
        e = np.array([3.0, 9.0])
        rows = g.gmres(inp.psi0, e, 0.5, 13.605, 1e-12, 20)
        g.haydock(inp.psi0, 30)
        again = g.haydock(inp.psi0, 12)
        assert np.array_equal(g.gmres(inp.psi0, e, 0.5, 13.605, 1e-12, 20), rows)
        for x, y in zip(first, again):
            assert np.array_equal(x, y)


def test_kept_workspaces_are_bounded_over_all_handles():
    """Eight handles whose solves take 216 MiB each: no more than 1 GiB of it stays with them
    (one more workspace if the runtime holds on to what was freed last, and 64 MiB for
    code and the handles' own small buffers)."""
    hip = C.CDLL("libamdhip64.so.7")  # the runtime the library already loaded

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    inp = synth.make_inputs(nb=8, kmesh=(16, 16, 16), xmesh=(2, 2, 2), lc=1, seed=97, xi_eV=3.0)
    gs = [core.OceanGPU.from_inputs(inp) for _ in range(8)]
    before = free()
    for g in gs:
        g.gmres(inp.psi0, np.array([3.0]), 0.5, 13.605, 1e-2, 15, return_status=True)
    used = before - free()
    print("kept", used, flush=True)
    assert used <= (1 << 30) + (216 << 20) + (64 << 20)
    want = gs[0].haydock(inp.psi0, 3)
    for g in gs[1:]:  # with and without a kept workspace
        for x, y in zip(g.haydock(inp.psi0, 3), want):
            assert np.array_equal(x, y)
    for g in gs:
        g.close()


def test_stacked_and_batched_planes_agree_with_interleaved():
    """ocean_gpu_haydock_multi and ocean_gpu_batch_haydock (host planes) against their
    interleaved forms, bit for bit; imag_a and niter_done may be null."""
    lib, n = core._lib(), 7
    inps = [synth.make_inputs(nb=9, kmesh=(3, 2, 4), xmesh=(3, 3, 3), lc=0, seed=98),
            synth.make_inputs(nb=13, kmesh=(2, 2, 2), xmesh=(3, 3, 3), lc=1, seed=99, xi_eV=3.0)]
    rng = np.random.default_rng(4)
    with core.OceanGPU.from_inputs(inps[0], nrhs=3) as g:
        psi = np.asfortranarray(rng.standard_normal(g.shape) + 1j * rng.standard_normal(g.shape)) / 30
        want = g.haydock_multi(psi, n)
        re, im = np.asfortranarray(psi.real), np.asfortranarray(psi.imag)
        a, b, ai = (np.zeros((3, n + 1)) for _ in range(3))
        done = np.zeros(3, np.int32)
        assert lib.ocean_gpu_haydock_multi(g.h, core._p(re), core._p(im), n, *(x.ctypes.data_as(core._DP) for x in (a, b, ai)),
                                           done.ctypes.data_as(core._IP)) == 0
        assert list(done) == [n] * 3 and all(np.array_equal(x, y) for x, y in zip((a, b, ai), want))
        assert lib.ocean_gpu_haydock_multi(g.h, core._p(re), core._p(im), n, a.ctypes.data_as(core._DP),
                                           b.ctypes.data_as(core._DP), None, None) == 0
        assert np.array_equal(a, want[0]) and np.array_equal(b, want[1])
    gs = [core.OceanGPU.from_inputs(i) for i in inps]
    bt = core.OceanBatch(gs)
    want, _ = bt.haydock([i.psi0 for i in inps], n)
    planes = [[np.asfortranarray(p) for p in (i.psi0.real, i.psi0.imag)] for i in inps]
    outs = [[np.zeros(n + 1) for _ in inps] for _ in range(3)]
    table = lambda arrays: (core._DP * 2)(*[x.ctypes.data_as(core._DP) for x in arrays])  # noqa: E731
    pr, pi = table([p[0] for p in planes]), table([p[1] for p in planes])
    done = np.zeros(2, np.int32)
    assert lib.ocean_gpu_batch_haydock(bt.b, pr, pi, n, *(table(o) for o in outs), done.ctypes.data_as(core._IP)) == 0
    assert list(done) == [n, n]
    for q in range(2):
        assert all(np.array_equal(o[q], w) for o, w in zip(outs, want[q]))
    assert lib.ocean_gpu_batch_haydock(bt.b, pr, None, n, *(table(o) for o in outs), None) == 1001
    bt.close()
    for g in gs:
        g.close()
