"""Krylov path on the GPU, through the C ABI (include/ucfdmat.h,
ucfdprecon.h, ucfdsolver.h), against the CPU oracle on the same seeded
inputs.

Bars: SpMV and the FP64 block LU-SGS apply are bit-exact (same operation
order, no FMA contraction); GMRES / BiCGSTAB follow the oracle step for step
with device dot products (fixed-order two-stage sums, so not bitwise equal to
the sequential CPU sum): same iteration counts and status, residual
histories within 1e-6 of max(|entry|, 1e-6 x initial residual), and the true
residual of the GPU solution within the requested tolerance.  The mixed apply (FP32 block products, FP64
diagonal LU) is within 1e-5 relative of the FP64 apply.
"""
import numpy as np
import pytest

from oracle import pyoracle as O
from ucfd_sparse_amd import layout as LY
from ucfd_sparse_amd import mesh as M

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def say(msg):
    print(f"[krylov-gpu] {msg}", flush=True)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def system(kind, size, seed, blk=5, colored=False):
    if kind == "tet":
        mesh = M.tet_mesh(size, seed=seed, permute=True)
    else:
        mesh = M.hex_mesh(*size, seed=seed, permute=True)
    flow = M.flow_fields(mesh, seed=seed)
    off = None
    if colored:
        lay = LY.colored_layout(mesh, flow)
        mesh, flow, off = lay.mesh, lay.flow, lay.off
    A = M.block_system(mesh, flow, blk=blk, seed=seed)
    return A, off


def dev_bsr(A):
    class D:
        pass
    d = D()
    d.bn, d.blk = A.bn, A.blk
    d.rowptr, d.colidx, d.diagslots = dev(A.rowptr), dev(A.colidx), dev(A.diagslots)
    d.values = dev(A.values)
    return d


@pytest.fixture(scope="module")
def K():
    from ucfd_sparse_amd import krylov
    return krylov


@pytest.fixture(scope="module")
def tet3():
    A, _ = system("tet", 3, 301)
    return A, M.normal_fill(A.bn * A.blk, 301), M.normal_fill(A.bn * A.blk, 302)


@pytest.mark.parametrize("blk", [1, 2, 3, 5, 7])
def test_spmv_device_bitwise(K, blk):
    say(f"BSR SpMV blk={blk}, device arrays")
    A, _ = system("tet", 4, 11, blk=blk)
    x = M.normal_fill(A.bn * blk, 12)
    y0 = M.normal_fill(A.bn * blk, 13)
    mat = K.SpMat.from_bsr(dev_bsr(A))
    yd = dev(y0)
    mat.mult(dev(x), yd, alpha=-1.0, beta=0.5)
    assert np.array_equal(yd.cpu().numpy(), O.spmv_bsr(A, x, -1.0, 0.5, y=y0))


def two_colour_dense(blk, nrow, per_row, seed):
    """A 2-colour BSR matrix with long rows: rows 0..nrow-1 (colour 0) couple
    only to rows nrow..2nrow-1 (colour 1) and back, per_row off-diagonal
    blocks per row, diagonally dominant.  One wave's rows then use more
    blocks than the LDS staging holds (multi-chunk SpMV, the HBM-direct path
    of the wave-staged sweeps)."""
    rng = np.random.default_rng(seed)
    bn = 2 * nrow
    rows, cols = [], []
    for i in range(bn):
        other = np.arange(nrow, bn) if i < nrow else np.arange(0, nrow)
        nb = np.sort(rng.choice(other, size=per_row, replace=False))
        c = np.sort(np.r_[nb, i])
        cols.append(c)
    rowptr = np.zeros(bn + 1, np.int32)
    rowptr[1:] = np.cumsum([len(c) for c in cols])
    colidx = np.concatenate(cols).astype(np.int32)
    diagslots = np.array([rowptr[i] + int(np.searchsorted(cols[i], i)) for i in range(bn)],
                         np.int32)
    values = rng.uniform(-0.1, 0.1, size=(len(colidx), blk, blk))
    for i in range(bn):
        values[diagslots[i]] += np.eye(blk) * (2.0 + per_row)
    return M.BSR(bn, blk, rowptr, colidx, diagslots, values), np.array([0, nrow, bn], np.int32)


@pytest.mark.parametrize("blk", [2, 5, 7])
def test_long_rows_spmv_and_colored_apply_bitwise(K, blk):
    say(f"long rows (14 blocks per row), blk={blk}: multi-chunk SpMV, HBM-direct sweeps")
    A, off = two_colour_dense(blk, 150, 13, 70 + blk)
    x = M.normal_fill(A.bn * blk, 71)
    y0 = M.normal_fill(A.bn * blk, 72)
    d = dev_bsr(A)
    mat = K.SpMat.from_bsr(d)
    yd = dev(y0)
    mat.mult(dev(x), yd, alpha=0.75, beta=-0.25)
    assert np.array_equal(yd.cpu().numpy(), O.spmv_bsr(A, x, 0.75, -0.25, y=y0))
    dv = O.blusgs_prepare(A)
    ref = O.blusgs_apply(A, dv, x, icolors=off)
    pc = K.Precon.from_bsr(d, icolors=off)
    bd = dev(x)
    pc.apply(bd)
    assert np.array_equal(bd.cpu().numpy(), ref)
    pc32 = K.Precon.from_bsr(d, icolors=off, fp32=True)
    bd = dev(x)
    pc32.apply(bd)
    err = np.abs(bd.cpu().numpy() - ref).max() / np.abs(ref).max()
    say(f"  mixed apply rel err {err:.2e}")
    assert err <= 1e-5


def test_spmv_host_arrays_staged(K, tet3):
    say("BSR SpMV, host arrays")
    A, b, x = tet3
    mat = K.SpMat.from_bsr(A)
    y = np.zeros(A.bn * A.blk)
    mat.mult(x, y, alpha=1.5)
    assert np.array_equal(y, O.spmv_bsr(A, x, 1.5, 0.0))


def test_csr_spmv_matches_blk1_oracle(K):
    say("CSR SpMV")
    A, _ = system("hex", (5, 4, 3), 21, blk=1)
    x = M.normal_fill(A.bn, 22)
    mat = K.SpMat(dev(A.rowptr), dev(A.colidx), dev(A.values.reshape(-1)), A.bn)
    y = dev(np.zeros(A.bn))
    mat.mult(dev(x), y, alpha=2.0)
    assert np.array_equal(y.cpu().numpy(), O.spmv_bsr(A, x, 2.0, 0.0))


def test_apply_sequential_level_scheduled_bitwise(K, tet3):
    say("sequential BLU-SGS apply (dependency levels)")
    A, b, _ = tet3
    pc = K.Precon.from_bsr(dev_bsr(A))
    bd = dev(b)
    pc.apply(bd)
    ref = O.blusgs_apply(A, O.blusgs_prepare(A), b)
    assert np.array_equal(bd.cpu().numpy(), ref)


def test_apply_colored_bitwise(K):
    say("coloured BLU-SGS apply, colour-ordered matrix")
    A, off = system("tet", 5, 41, colored=True)
    b = M.normal_fill(A.bn * A.blk, 42)
    pc = K.Precon.from_bsr(dev_bsr(A), icolors=off)
    bd = dev(b)
    pc.apply(bd)
    dv = O.blusgs_prepare(A)
    ref = O.blusgs_apply(A, dv, b, icolors=off)
    assert np.array_equal(bd.cpu().numpy(), ref)
    assert np.array_equal(ref, O.blusgs_apply(A, dv, b))


def test_apply_colored_with_coupled_ranges_bitwise(K, tet3):
    """Colour ranges that couple internally: the rows of each range run in
    the reference's one-thread order (dependency levels inside the range)."""
    say("coloured apply, internally coupled ranges")
    A, b, _ = tet3
    off = np.array([0, A.bn // 3, A.bn // 2, A.bn], np.int32)
    pc = K.Precon.from_bsr(dev_bsr(A), icolors=off)
    bd = dev(b)
    pc.apply(bd)
    ref = O.blusgs_apply(A, O.blusgs_prepare(A), b, icolors=off)
    assert np.array_equal(bd.cpu().numpy(), ref)


def test_apply_host_arrays(K, tet3):
    say("sequential apply, host arrays")
    A, b, _ = tet3
    pc = K.Precon.from_bsr(A)
    bh = b.copy()
    pc.apply(bh)
    assert np.array_equal(bh, O.blusgs_apply(A, O.blusgs_prepare(A), b))


@pytest.mark.parametrize("colored", [False, True])
def test_apply_mixed_precision_close(K, colored):
    say(f"mixed FP32/FP64 apply, colored={colored}")
    A, off = system("tet", 5, 51, colored=colored)
    b = M.normal_fill(A.bn * A.blk, 52)
    pc = K.Precon.from_bsr(dev_bsr(A), icolors=off if colored else None, fp32=True)
    bd = dev(b)
    pc.apply(bd)
    got = bd.cpu().numpy()
    ref = O.blusgs_apply(A, O.blusgs_prepare(A), b, icolors=off if colored else None)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    say(f"  rel err {err:.2e}")
    assert np.all(np.isfinite(got))
    assert 0 < err <= 1e-5


def _close_hist(h_gpu, h_orc, n):
    """Largest history difference relative to max(|entry|, 1e-6 * first
    entry): residuals near the convergence floor are differences of nearly
    equal numbers, compared against the scale of the problem."""
    h_gpu, h_orc = np.asarray(h_gpu[:n]), np.asarray(h_orc[:n])
    if n == 0:
        return 0.0
    scale = np.maximum(np.abs(h_orc), 1e-6 * abs(h_orc[0]))
    return float((np.abs(h_gpu - h_orc) / scale).max())


@pytest.mark.parametrize("precon", [True, False])
def test_gmres_left_matches_oracle(K, tet3, precon):
    say(f"GMRES(5) left-preconditioned, precon={precon}")
    A, b, _ = tet3
    tol, m, maxiter = (1e-10, 5, 40) if precon else (1e-9, 4, 60)
    xo, ito, sto, reso, histo = O.gmres(A, b, m=m, maxiter=maxiter, tol=tol, precon=precon)
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    pc = K.Precon.from_bsr(D) if precon else K.Precon.none()
    s = K.Solver("gmres", A.bn * A.blk, maxiter, tol, m=m)
    x = dev(np.zeros(A.bn * A.blk))
    st, it, res = s.solve(pc, mat, x, dev(b))
    say(f"  gpu it={it} st={st} res={res:.3e}; oracle it={ito} st={sto} res={reso:.3e}")
    assert (it, st) == (ito, sto)
    assert _close_hist(s.history(), histo, it + 1 if it < maxiter else it) <= 1e-6
    xg = x.cpu().numpy()
    assert np.linalg.norm(b - A.to_scipy() @ xg) <= 10 * tol
    assert np.allclose(xg, xo, rtol=1e-6, atol=1e-9 * np.abs(xo).max())


def test_gmres_long_restart_matches_oracle(K, tet3):
    """One full cycle of GMRES(40) without a preconditioner: the Arnoldi
    steps project onto 1 .. 40 basis vectors, so the projection kernels run
    at every register width (8, 16, 32 columns) and past 32 (separate
    passes); the solution follows the oracle's (true residual 3.5e-9 of
    |b| = 29)."""
    say("GMRES(40), one full cycle")
    A, b, _ = tet3
    m, maxiter, tol = 40, 1, 1e-30
    xo, ito, sto, reso, histo = O.gmres(A, b, m=m, maxiter=maxiter, tol=tol, precon=False)
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    s = K.Solver("gmres", A.bn * A.blk, maxiter, tol, m=m)
    x = dev(np.zeros(A.bn * A.blk))
    st, it, res = s.solve(K.Precon.none(), mat, x, dev(b))
    say(f"  gpu it={it} st={st} res={res:.3e}; oracle it={ito} st={sto} res={reso:.3e}")
    assert (it, st) == (ito, sto) == (maxiter, st)
    assert _close_hist(s.history(), histo, it) <= 1e-6
    xg = x.cpu().numpy()
    assert np.linalg.norm(b - A.to_scipy() @ xg) <= 1e-8
    assert np.allclose(xg, xo, rtol=1e-6, atol=1e-9 * np.abs(xo).max())


@pytest.mark.parametrize("precon", [True, False])
def test_bicgstab_matches_oracle(K, tet3, precon):
    say(f"BiCGSTAB, precon={precon}")
    A, b, _ = tet3
    tol, maxiter = (1e-10, 60) if precon else (1e-9, 80)
    xo, ito, sto, reso, histo = O.bicgstab(A, b, maxiter=maxiter, tol=tol, precon=precon)
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    pc = K.Precon.from_bsr(D) if precon else K.Precon.none()
    s = K.Solver("bicgstab", A.bn * A.blk, maxiter, tol)
    x = dev(np.zeros(A.bn * A.blk))
    st, it, res = s.solve(pc, mat, x, dev(b))
    say(f"  gpu it={it} st={st} res={res:.3e}; oracle it={ito} st={sto} res={reso:.3e}")
    assert (it, st) == (ito, sto)
    assert _close_hist(s.history(), histo, it + 1) <= 1e-6
    xg = x.cpu().numpy()
    assert np.linalg.norm(b - A.to_scipy() @ xg) <= 1e-8
    assert np.allclose(xg, xo, rtol=1e-6, atol=1e-9 * np.abs(xo).max())


@pytest.mark.parametrize("kind", ["gmres", "bicgstab"])
def test_right_preconditioned_mixed_reaches_rtol(K, kind):
    """The Krylov workload's form: right-preconditioned by the coloured
    block LU-SGS with the FP32 apply, FP64 Krylov, rtol 1e-10."""
    say(f"{kind} right/relative, coloured FP32 apply, 12^3x6 tets")
    A, off = system("tet", 12, 61, colored=True)
    b = M.normal_fill(A.bn * A.blk, 62)
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    pc = K.Precon.from_bsr(D, icolors=off, fp32=True)
    s = K.Solver(kind, A.bn * A.blk, 200, 1e-10, m=30, right=True)
    x = dev(np.zeros(A.bn * A.blk))
    st, it, res = s.solve(pc, mat, x, dev(b))
    rel = np.linalg.norm(b - A.to_scipy() @ x.cpu().numpy()) / np.linalg.norm(b)
    say(f"  it={it} st={st} true rel residual {rel:.2e}")
    assert st == 0
    assert rel <= 1e-9
    if kind == "gmres":
        xo, ito, sto, _, _ = O.gmres(A, b, m=30, maxiter=200, tol=1e-10, right=True,
                                     icolors=off)
        assert sto == 0
        assert np.allclose(x.cpu().numpy(), xo, rtol=1e-7, atol=1e-8 * np.abs(xo).max())


def test_solves_are_deterministic(K, tet3):
    say("determinism of two GMRES solves")
    A, b, _ = tet3
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    pc = K.Precon.none()
    out = []
    for _ in range(2):
        s = K.Solver("gmres", A.bn * A.blk, 30, 1e-9, m=4)
        x = dev(np.zeros(A.bn * A.blk))
        s.solve(pc, mat, x, dev(b))
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0], out[1])


def test_status_codes(K, tet3):
    say("solver status codes")
    A, b, _ = tet3
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    pc = K.Precon.none()
    s = K.Solver("gmres", A.bn * A.blk, 1, 1e-14, m=2)
    st, it, _ = s.solve(pc, mat, dev(np.zeros(A.bn * A.blk)), dev(b))
    assert (st, it) == (K.REACH_ITERMAX, 1)
    s2 = K.Solver("bicgstab", A.bn * A.blk, 5, 1e-10)
    st, it, _ = s2.solve(pc, mat, dev(np.zeros(A.bn * A.blk)), dev(np.zeros(A.bn * A.blk)))
    assert (st, it) == (K.RHOBREAKDOWN, 0)


@pytest.mark.parametrize("bn", [1000, 40_000])
def test_pi_breakdown_leaves_x(K, bn):
    """BiCGSTAB with rt.(A p) = 0 in the first iteration (skew blocks, a residual of
    equal entries): the breakdown status, and x as it was, where the kernels sum
    the partials of a reduction themselves (8 of them) and where a launch of its
    own does (313)."""
    say(f"pi breakdown, {bn} blocks")
    rng = np.random.default_rng(bn)
    rows = np.arange(bn + 1, dtype=np.int32)
    mat = K.SpMat(dev(rows), dev(rows[:-1]), dev(np.tile([0.0, 1.0, -1.0, 0.0], bn)), bn, 2)
    x0 = rng.integers(-9, 10, 2 * bn).astype(np.float64)    # every sum below is exact
    r = np.repeat(rng.integers(1, 8, bn), 2).astype(np.float64)
    b = r + np.stack([x0[1::2], -x0[::2]], 1).reshape(-1)
    s = K.Solver("bicgstab", 2 * bn, 5, 1e-10)
    for _ in range(2):
        x = dev(x0)
        st, it, _ = s.solve(K.Precon.none(), mat, x, dev(b))
        assert (st, it) == (K.PIBREAKDOWN, 0)
        assert np.array_equal(x.cpu().numpy(), x0)


def test_errors_are_reported_not_faulted(K, tet3):
    say("index and pivot errors")
    from ucfd_sparse_amd import lib as L
    A, b, x = tet3
    bad = A.colidx.copy()
    bad[7] = A.bn + 5
    mat = K.SpMat(dev(A.rowptr), dev(bad), dev(A.values), A.bn, A.blk)
    with pytest.raises(L.UCFDError):
        mat.mult(dev(x), dev(np.zeros(A.bn * A.blk)))
    with pytest.raises(L.UCFDError):
        K.Precon(dev(A.rowptr), dev(bad), dev(A.diagslots), dev(A.values), A.bn, A.blk)
    vals = A.values.copy()
    vals[A.diagslots[3]] = 0.0
    with pytest.raises(L.UCFDError):
        K.Precon(dev(A.rowptr), dev(A.colidx), dev(A.diagslots), dev(vals), A.bn, A.blk)
    # the library keeps working after the errors
    ok = K.SpMat.from_bsr(dev_bsr(A))
    y = dev(np.zeros(A.bn * A.blk))
    ok.mult(dev(x), y)
    assert np.array_equal(y.cpu().numpy(), O.spmv_bsr(A, x))


def test_c_abi_program_matches_oracle():
    """tests/abi/krylov_calls.c: the reference's call sequence from C on host
    arrays; every result compared with the oracle."""
    import os
    import subprocess
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = os.path.join(repo, "tests", "abi", "krylov_calls.x")
    if not os.path.exists(exe):
        pytest.fail("tests/abi/krylov_calls.x not built (run __graft_entry__.build())")
    out = os.path.join(repo, "gpurun_out", "krylov_calls.bin")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    say("C caller krylov_calls.x bn=40")
    r = subprocess.run([exe, out, "40"], capture_output=True, text=True, timeout=120)
    say(r.stdout.strip())
    assert r.returncode == 0, r.stderr
    raw = open(out, "rb").read()
    pos = 0

    def take(dtype, count):
        nonlocal pos
        sz = count * np.dtype(dtype).itemsize
        a = np.frombuffer(raw[pos:pos + sz], dtype)
        pos += sz
        return a
    bn, blk, nnz, nc = take(np.int32, 4)
    n = bn * blk
    icolors = take(np.int32, nc + 1)
    A = M.BSR(int(bn), int(blk), take(np.int32, bn + 1).copy(), take(np.int32, nnz).copy(),
              take(np.int32, bn).copy(), take(np.float64, nnz * blk * blk).reshape(nnz, blk, blk)
              .copy())
    x, b = take(np.float64, n), take(np.float64, n)
    assert np.array_equal(take(np.float64, n), O.spmv_bsr(A, x, 1.5, 0.0))
    dv = O.blusgs_prepare(A)
    ref = O.blusgs_apply(A, dv, b)
    assert np.array_equal(take(np.float64, n), ref)
    assert np.array_equal(take(np.float64, n), O.blusgs_apply(A, dv, b, icolors=icolors))
    for kind in ("gmres", "bicgstab"):
        xs = take(np.float64, n)
        it, st = take(np.int32, 2)
        res = take(np.float64, 1)[0]
        hist = take(np.float64, 30)
        if kind == "gmres":
            xo, ito, sto, reso, histo = O.gmres(A, b, m=4, maxiter=30, tol=1e-10)
        else:
            xo, ito, sto, reso, histo = O.bicgstab(A, b, maxiter=30, tol=1e-10)
        say(f"  {kind}: C it={it} st={st} res={res:.3e}; oracle it={ito} st={sto}")
        assert (it, st) == (ito, sto)
        assert _close_hist(hist, histo, min(int(it) + 1, 30)) <= 1e-6
        assert np.allclose(xs, xo, rtol=1e-6, atol=1e-9 * np.abs(xo).max())


def diagonal_bsr(bn, blk, seed):
    rng = np.random.default_rng(seed)
    rowptr = np.arange(bn + 1, dtype=np.int32)
    colidx = np.arange(bn, dtype=np.int32)
    values = rng.uniform(-0.2, 0.2, size=(bn, blk, blk)) + np.eye(blk) * 3.0
    return M.BSR(bn, blk, rowptr, colidx, rowptr[:-1].copy(), values)


@pytest.mark.parametrize("blk", [1, 5])
def test_block_diagonal_matrix_closed_forms(K, blk):
    """Rows without off-diagonal blocks (nothing staged by the wave kernels):
    SpMV = D x, both preconditioners apply D^-1 exactly (= the oracle's LU
    solve), and the preconditioned solvers stop at the first check."""
    say(f"block-diagonal matrix, blk={blk}")
    A = diagonal_bsr(700, blk, 80 + blk)
    x = M.normal_fill(A.bn * blk, 81)
    D = dev_bsr(A)
    mat = K.SpMat.from_bsr(D)
    y = dev(np.zeros(A.bn * blk))
    mat.mult(dev(x), y)
    assert np.array_equal(y.cpu().numpy(), O.spmv_bsr(A, x))
    dinv = O.blusgs_apply(A, O.blusgs_prepare(A), x)
    for icolors in (None, np.array([0, A.bn], np.int32)):
        pc = K.Precon.from_bsr(D, icolors=icolors)
        b = dev(x)
        pc.apply(b)
        assert np.array_equal(b.cpu().numpy(), dinv)
    D2 = dev_bsr(A)
    pcb = K.Precon.from_bsr(D2, kind="bilu")
    b = dev(x)
    pcb.apply(b)
    f = O.ilu_prepare(A, "bilu")
    assert np.array_equal(b.cpu().numpy(), O.ilu_apply(A, f, x, "bilu"))
    for kind in ("gmres", "bicgstab"):
        s = K.Solver(kind, A.bn * blk, 10, 1e-10, m=5)
        xs = dev(np.zeros(A.bn * blk))
        st, it, res = s.solve(K.Precon.from_bsr(D), mat, xs, dev(x))
        ref = O.gmres(A, x, 5, 10, 1e-10) if kind == "gmres" else O.bicgstab(A, x, 10, 1e-10)
        say(f"  {kind}: status {st}, iterations {it}, residual {res:.2e}; oracle {ref[2]}, {ref[1]}")
        assert (it, st) == (ref[1], ref[2])
        assert np.linalg.norm(x - A.to_scipy() @ xs.cpu().numpy()) <= 1e-9 * np.linalg.norm(x)


def test_ragged_rows_bitwise(K):
    """A matrix whose rows range from diagonal-only to many blocks: SpMV and
    the sequential and block-ILU applies bit for bit against the oracle."""
    import sys as _s
    import os as _o
    _s.path.insert(0, _o.path.join(_o.path.dirname(_o.path.abspath(__file__)), "golden"))
    import make_golden
    say("ragged rows")
    A = make_golden.random_pattern_bsr(500, 3, 3, 93)
    deg = np.diff(A.rowptr)
    assert deg.min() == 1 and deg.max() >= 6
    x = M.normal_fill(A.bn * 3, 94)
    D = dev_bsr(A)
    y = dev(np.zeros(A.bn * 3))
    K.SpMat.from_bsr(D).mult(dev(x), y)
    assert np.array_equal(y.cpu().numpy(), O.spmv_bsr(A, x))
    b = dev(x)
    K.Precon.from_bsr(D).apply(b)
    assert np.array_equal(b.cpu().numpy(), O.blusgs_apply(A, O.blusgs_prepare(A), x))
    D2 = dev_bsr(A)
    b = dev(x)
    K.Precon.from_bsr(D2, kind="bilu").apply(b)
    assert np.array_equal(b.cpu().numpy(), O.ilu_apply(A, O.ilu_prepare(A, "bilu"), x, "bilu"))


def test_prepare_again_with_new_values(K):
    """A later Prepare reuses the schedule built by the first and reads only
    the values: after the values change in place, the apply equals the
    oracle's on the new values (block LU-SGS and coloured block ILU(0))."""
    say("second Prepare on new values")
    A, off = system("tet", 4, 95, colored=True)
    x = M.normal_fill(A.bn * A.blk, 96)
    D = dev_bsr(A)
    pc = K.Precon.from_bsr(D, icolors=off)
    rng = np.random.default_rng(97)
    A2 = M.BSR(A.bn, A.blk, A.rowptr, A.colidx, A.diagslots,
               A.values * rng.uniform(0.9, 1.1, size=A.values.shape))
    D.values.copy_(dev(A2.values))
    pc.prepare()
    b = dev(x)
    pc.apply(b)
    assert np.array_equal(b.cpu().numpy(), O.blusgs_apply(A2, O.blusgs_prepare(A2), x, icolors=off))
    Di = dev_bsr(A)
    pci = K.Precon.from_bsr(Di, icolors=off, kind="bilu")
    Di.values.copy_(dev(A2.values))
    pci.prepare()
    b = dev(x)
    pci.apply(b)
    f = O.ilu_prepare(A2, "pbilu")
    assert np.array_equal(Di.values.cpu().numpy(), f.reshape(A.values.shape))
    assert np.array_equal(b.cpu().numpy(), O.ilu_apply(A2, f, x, "pbilu", off))


@pytest.mark.parametrize("dims", [(3, 17, 257), (4, 29, 113)])
@pytest.mark.parametrize("kind", ["gmres", "bicgstab"])
def test_solves_on_both_sides_of_the_reduction_choice(K, dims, kind):
    """65535 and 65540 unknowns: 256 partials a row (summed by the kernel that
    uses them) and 257 (summed to one value first)."""
    mesh = M.hex_mesh(*dims, seed=13)
    A = M.block_system(mesh, M.flow_fields(mesh, seed=13), blk=5, seed=13)
    b = M.normal_fill(A.bn * 5, 13)
    x = np.zeros_like(b)
    s = K.Solver(kind, A.bn * 5, 200, 1e-10, m=30, right=True)
    status, _, _ = s.solve(K.Precon.from_bsr(A), K.SpMat.from_bsr(A), x, b)
    assert status == K.CONVERGED
    r = b - A.to_scipy() @ x
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b)
