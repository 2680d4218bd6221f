"""Differentiation form on the GPU: the adjoint kernels (ucfd_lusgs_adjoint)
against the CPU adjoint oracle on the same inputs, and the
torch.autograd.Function (ucfd_sparse_amd.autograd.LUSGSPass) against central
differences of the GPU forward (h = 1e-6, FP64), with dQ* stored and
recomputed (identical gradients)."""
import ctypes
import math

import numpy as np
import pytest

from oracle import pyoracle as O
from ucfd_sparse_amd import layout as LY
from ucfd_sparse_amd import lib as L
from ucfd_sparse_amd import mesh as M

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SCALE = {"rhsb": 1.0, "dt": 1.0, "fspr": 1e3}   # see tests/test_adjoint_oracle.py


def say(msg):
    print(f"[adjoint-gpu] {msg}", flush=True)


@pytest.fixture(scope="module")
def setup():
    from ucfd_sparse_amd.autograd import ColoredSystem
    mesh = M.tet_mesh(5, seed=19, permute=True)
    flow = M.flow_fields(mesh, seed=19)
    lay = LY.colored_layout(mesh, flow)
    S = ColoredSystem(lay)
    yield lay, S
    S.close()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_adjoint_kernels_match_oracle(setup):
    lay, S = setup
    m, f = lay.mesh, lay.flow
    say(f"adjoint vs oracle, {m.neles} cells, {lay.ncolors} colours")
    rng = np.random.default_rng(5)
    w = rng.normal(size=(5, m.neles))
    rhs, dt, fspr = dev(f.rhsb[:5]), dev(f.dt), dev(f.fspr)
    dq, dstar, _ = S.forward_arrays(rhs, dt, fspr)
    torch.cuda.synchronize()
    od, ods, odq, _ = O.colored_pass(m.nei_ele, lay.icolor, lay.lcolor, m.fnorm_vol, m.vec_fnorm,
                                     f.fspr, f.dt, f.upts, f.rhsb)
    assert np.array_equal(dq.cpu().numpy(), odq)
    assert np.array_equal(dstar.cpu().numpy(), ods)
    rb, dtb, fb = S.adjoint(dt, fspr, dstar, dq, dev(w))
    torch.cuda.synchronize()
    orb, odtb, ofb = O.lusgs_adjoint(m.nei_ele, lay.off, m.fnorm_vol, m.vec_fnorm, f.fspr, f.dt,
                                     f.upts, ods, odq, w)
    for name, g, o in (("rhsbar", rb, orb), ("dtbar", dtb, odtb), ("fsprbar", fb, ofb)):
        g = g.cpu().numpy()
        diff = np.abs(g - o).max() / np.abs(o).max()
        say(f"  {name}: bitwise={np.array_equal(g, o)} max rel diff {diff:.1e}")
        assert diff <= 1e-13


@pytest.mark.parametrize("recompute", [False, True])
def test_autograd_matches_central_differences(setup, recompute):
    from ucfd_sparse_amd.autograd import lusgs_pass
    lay, S = setup
    m, f = lay.mesh, lay.flow
    say(f"autograd vs central differences, recompute={recompute}")
    rng = np.random.default_rng(7)
    w = dev(rng.normal(size=(5, m.neles)))
    rhs = dev(f.rhsb[:5]).requires_grad_()
    dt = dev(f.dt).requires_grad_()
    fspr = dev(f.fspr).requires_grad_()
    J = (w * lusgs_pass(S, rhs, dt, fspr, recompute=recompute)).sum()
    J.backward()
    grads = {"rhsb": rhs.grad, "dt": dt.grad, "fspr": fspr.grad}
    base = {"rhsb": rhs.detach(), "dt": dt.detach(), "fspr": fspr.detach()}

    def Jof(**kw):
        x = dict(base, **kw)
        dq, _, _ = S.forward_arrays(x["rhsb"], x["dt"], x["fspr"])
        return math.fsum((w * dq).double().cpu().numpy().ravel())
    h = 1e-6
    worst = {}
    for name in ("rhsb", "dt", "fspr"):
        for k in range(8):
            d = torch.from_numpy(rng.normal(size=tuple(base[name].shape)) * SCALE[name]).cuda()
            fd = (Jof(**{name: base[name] + h * d}) - Jof(**{name: base[name] - h * d})) / (2 * h)
            ad = float((grads[name] * d).sum())
            worst[name] = max(worst.get(name, 0.0), abs(fd - ad) / abs(ad))
    say(f"  worst relative FD disagreement {worst}")
    assert max(worst.values()) <= 1e-6
    if recompute:
        rhs2 = base["rhsb"].clone().requires_grad_()
        dt2 = base["dt"].clone().requires_grad_()
        fs2 = base["fspr"].clone().requires_grad_()
        (w * lusgs_pass(S, rhs2, dt2, fs2, recompute=False)).sum().backward()
        assert torch.equal(rhs2.grad, rhs.grad)
        assert torch.equal(dt2.grad, dt.grad)
        assert torch.equal(fs2.grad, fspr.grad)


def test_non_coloured_layout_is_rejected():
    import ctypes

    from ucfd_sparse_amd import lib as L
    mesh = M.tet_mesh(3, seed=3, permute=True)
    nei = dev(mesh.nei_ele)
    h = ctypes.c_void_p()
    off = np.array([0, mesh.neles], np.int32)
    lib = L.load()
    assert lib.ucfd_adjoint_create.argtypes is not None
    rc = lib.ucfd_adjoint_create(ctypes.byref(h), mesh.neles, mesh.nface, 1, off.ctypes.data,
                                 nei.data_ptr(), None, None, None)
    assert rc != 0


@pytest.mark.parametrize("coloring", ["greedy", "greedy-bfs"])
def test_one_call_pass_equals_the_separate_calls(coloring):
    """ucfd_lusgs_pass (both forms, and the lower half alone) against
    parallel_pre_lusgs and the per-colour sweep calls, bit for bit."""
    from ucfd_sparse_amd.autograd import ColoredSystem
    L.call("ucfd_set_config", 5, 5, 3)
    mesh = M.tet_mesh(6, seed=4)
    lay = LY.colored_layout(mesh, M.flow_fields(mesh, seed=4), coloring=coloring)
    S = ColoredSystem(lay)
    rhsb, dt, fspr = (torch.from_numpy(a).cuda() for a in (lay.flow.rhsb, lay.flow.dt,
                                                           lay.flow.fspr))
    diag, dstar, dq = torch.zeros_like(dt), torch.zeros_like(rhsb), torch.zeros_like(rhsb)
    mesh_args = (S.N, S.F, S.nei, S.icolor, S.lcolor, S.fnv, S.vfn, S.upts)
    L.call("parallel_pre_lusgs", S.N, S.F, 1.5, S.fnv, dt, diag, fspr)
    for c in range(len(S.off) - 1):
        L.call("ns_parallel_lower_sweep", S.off[c], S.off[c + 1], *mesh_args, rhsb, dstar, diag,
               fspr)
    for c in reversed(range(len(S.off) - 1)):
        L.call("ns_parallel_upper_sweep", S.off[c], S.off[c + 1], *mesh_args, dq, dstar, diag, fspr)
    got = S.forward_arrays(rhsb, dt, fspr, 1.5)
    assert all(torch.equal(g, w) for g, w in zip(got, (dq, dstar, diag)))
    assert torch.equal(S.forward_inplace(rhsb, dt, fspr, 1.5), dq)
    assert torch.equal(S.recompute_dstar(rhsb, dt, fspr, 1.5), dstar)
    with pytest.raises(L.UCFDError):
        S.nei[2, 5] = S.N + 3
        S.forward_arrays(rhsb, dt, fspr)
    S.nei[2, 5] = 5
    S.forward_arrays(rhsb, dt, fspr)        # the raised error was cleared


@pytest.mark.parametrize("kind,dims", [("hex", (5, 5, 5)), ("hex", (4, 4, 8)), ("hex", (13, 5, 2)),
                                       ("quad", (13, 10, 1)), ("quad", (9, 7, 1)), ("tet", (4,))])
def test_adjoint_at_workgroup_edges(kind, dims):
    """Colours of 62 to 65 cells (one 64-cell workgroup, just under and just
    over) and every face count the meshes have, against the adjoint oracle."""
    mesh = M.tet_mesh(*dims, seed=9) if kind == "tet" else M.hex_mesh(*dims, seed=9)
    if kind == "quad":
        mesh = M.Mesh(np.ascontiguousarray(mesh.nei_ele[:4]),
                      np.ascontiguousarray(mesh.fnorm_vol[:4]),
                      np.ascontiguousarray(mesh.vec_fnorm[:4, :2]), mesh.orig_id, mesh.key)
    lay = LY.colored_layout(mesh, M.flow_fields(mesh, seed=9), coloring="greedy-bfs")
    m, f = lay.mesh, lay.flow
    N, F, D = m.neles, m.nface, m.ndims
    rng = np.random.default_rng(9)
    w = rng.normal(size=(D + 2, N))
    _, ds, dq, _ = O.colored_pass(m.nei_ele, lay.icolor, lay.lcolor, m.fnorm_vol, m.vec_fnorm,
                                  f.fspr, f.dt, f.upts, f.rhsb)
    want = O.lusgs_adjoint(m.nei_ele, lay.off, m.fnorm_vol, m.vec_fnorm, f.fspr, f.dt, f.upts, ds,
                           dq, w)
    off = np.ascontiguousarray(lay.off, np.int32)
    mesh_d = [dev(a) for a in (m.nei_ele, m.fnorm_vol, m.vec_fnorm, f.upts)]
    dt, fspr, dqd, wd = dev(f.dt), dev(f.fspr), dev(dq), dev(w)
    dtb, fb, h = torch.zeros_like(dt), torch.zeros_like(fspr), ctypes.c_void_p()
    L.call("ucfd_set_config", D + 2, D + 2, D)
    try:
        L.call("ucfd_adjoint_create", h, N, F, len(off) - 1, off, *mesh_d)
        for alias in (False, True):
            dsd = dev(ds)
            rb = dsd if alias else torch.zeros_like(dsd)
            L.call("ucfd_lusgs_adjoint", h.value, 1.0, dt, fspr, dsd, dqd, wd, rb, dtb, fb)
            for g, o, what in zip((rb, dtb, fb), want, ("rhsb", "dt", "fspr")):
                assert np.abs(g.cpu().numpy() - o).max() <= 1e-13 * np.abs(o).max(), (what, alias)
    finally:
        L.load().ucfd_adjoint_destroy(h)
        L.call("ucfd_set_config", 5, 5, 3)
