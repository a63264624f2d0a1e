"""GPU parity of the plain column solvers, through the C-ABI, against the oracle.

FP64 Thomas kernels follow the reference operation order without FMA
contraction, so they must agree with the oracle to within a few ulps
(tolerance 1e-14 relative, well inside the 1e-12 drop-in bar).  PCR and the
mixed-precision solver use a different elimination order; their tolerances
are stated per test.
"""
import numpy as np
import pytest

from helpers import diag_dominant_system, gpu_available, relerr

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def torch_dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def config1_system(rng, ncol, nk):
    """5 deg dt-shaped system: a,c = -U(0.5,2); b = -(a+c)+U(0.1,1); Dirichlet
    bottom through the ghost row (q(1) -= p(1), f(1) -= 2 p(1) T_lbc, p(1) = 0)
    and r(top) = 0 (dt_ng.F90:147-163); rhs = 1000-800 exp(-(z+7)/2) + N(0,5)."""
    a, b, c = diag_dominant_system(rng, ncol, nk)
    z = -7. + 0.5 * np.arange(nk)
    f = 1000. - 800. * np.exp(-(z + 7.) / 2.) + rng.normal(0., 5., size=(ncol, nk))
    tlbc = 181. + rng.normal(0., 1., size=ncol)
    b[:, 0] -= a[:, 0]
    f[:, 0] -= 2. * a[:, 0] * tlbc
    a[:, 0] = 0.
    c[:, nk - 2] = 0.
    return a, b, c, f


def test_trsolv_dropin_config1_per_latitude(pkg, oracle):
    # dt.F:330 calls trsolv per latitude: lev0..lev1 = 1..29, rows 1..28,
    # lon0..lon1 = 1..76 (nlonp4 = 76, periodic columns skipped); every one
    # of the 5 degree grid's 36 latitudes, as one step of the model calls it.
    rng = np.random.default_rng(0x7E6C0000)
    nlev, nlonp4 = 29, 76
    for lat in range(1, 37):
        a, b, c, f = config1_system(rng, nlonp4, nlev)
        x = np.full((nlonp4, nlev), 1e30)
        y = x.copy()
        pkg.tgx.trsolv(a, b, c, f, x, 1, nlev, 1, nlev - 1, 1, nlonp4, nlonp4, lat, 0)
        oracle.trsolv(a, b, c, f, y, 1, nlev, 1, nlev - 1, 1, nlonp4, nlonp4)
        assert np.array_equal(x[:, nlev - 1], y[:, nlev - 1])   # untouched row
        assert np.array_equal(x[:2], y[:2]) and np.array_equal(x[-2:], y[-2:])
        assert relerr(x, y) <= 1e-14, relerr(x, y)


@pytest.mark.parametrize("name,k2off", [("g5", 1), ("g2p5", 0), ("nest1", 1)])
def test_trsolv_ng_dropin(pkg, oracle, name, k2off):
    g = pkg.synth.make_grid(name)
    nk, nlond, nlatd = g["nk"], g["nlon"] + 4, g["nlat"] + 4
    rng = np.random.default_rng(g["seed"])
    a, b, c, f = config1_system(rng, nlond * nlatd, nk)
    shp = (nlatd, nlond, nk)
    a, b, c, f = (np.ascontiguousarray(v.reshape(shp)) for v in (a, b, c, f))
    k2 = nk - k2off
    x = np.zeros(shp)
    y = np.zeros(shp)
    pkg.tgx.trsolv_ng(a, b, c, f, x, k2)
    oracle.trsolv_ng(a, b, c, f, y, nk, nlond * nlatd, k2)
    assert relerr(x[..., :k2], y[..., :k2]) <= 1e-14


def test_blktri_dropin(pkg, oracle):
    from test_oracle_solvers import random_blocks, to_colmajor
    rng = np.random.default_rng(11)
    ncol, nlev, nlonp4 = 76, 57, 76
    P, Q, R, F = random_blocks(rng, ncol, nlev, 2)
    args = [to_colmajor(P), to_colmajor(Q), to_colmajor(R), np.ascontiguousarray(F)]
    x = np.zeros((ncol, nlev, 2))
    y = np.zeros((ncol, nlev, 2))
    pkg.tgx.blktri(*args, x, 1, nlev, 1, nlonp4, nlonp4)
    oracle.blktri(*args, y, 1, nlev, 1, nlonp4, nlonp4)
    assert np.array_equal(x[:2], y[:2]) and np.array_equal(x[-2:], y[-2:])
    assert relerr(x, y) <= 1e-14


def test_blktri3_dropin(pkg, oracle):
    from test_oracle_solvers import random_blocks, to_colmajor
    rng = np.random.default_rng(12)
    ncol, nk = 300, 57
    P, Q, R, F = random_blocks(rng, ncol, nk, 3)
    args = [to_colmajor(P), to_colmajor(Q), to_colmajor(R), np.ascontiguousarray(F)]
    x = np.zeros((ncol, nk, 3))
    y = np.zeros((ncol, nk, 3))
    pkg.tgx.blktri3(*args, x, nk - 1)
    oracle.blktri3(*args, y, nk, ncol, nk - 1)
    assert relerr(x, y) <= 1e-14


@pytest.mark.parametrize("nk", [29, 57, 113, 200])
@pytest.mark.parametrize("scheme", [1, 2, 0])
def test_trsolv_dev_schemes(pkg, oracle, nk, scheme):
    import torch
    rng = np.random.default_rng(nk + 100 * scheme)
    ncol = 4099
    a, b, c, f = config1_system(rng, ncol, nk)
    k2 = nk - 2
    y = np.zeros((ncol, nk))
    oracle.trsolv_ng(a, b, c, f, y, nk, ncol, k2)
    da, db, dc, df = (torch_dev(v) for v in (a, b, c, f))
    dx = torch.full((ncol, nk), -1.0, dtype=torch.float64, device="cuda")
    pkg.tgx.trsolv_dev(da, db, dc, df, dx, 0, k2 - 1, scheme=scheme)
    torch.cuda.synchronize()
    x = dx.cpu().numpy()
    tol = 1e-14 if scheme == 1 else 1e-12
    assert relerr(x[:, :k2], y[:, :k2]) <= tol
    assert np.all(x[:, k2:] == -1.0)
    if scheme == 0:
        assert pkg.tgx.autotune_choice(nk, 0, k2 - 1, ncol) in (1, 2)


@pytest.mark.parametrize("nsweep,tol", [(0, 1e-5), (1, 1e-9), (2, 1e-10)])
def test_trsolv_mixed_precision(pkg, oracle, nsweep, tol):
    import torch
    rng = np.random.default_rng(77 + nsweep)
    ncol, nk = 8192, 113
    a, b, c, f = config1_system(rng, ncol, nk)
    y = np.zeros((ncol, nk))
    oracle.trsolv_ng(a, b, c, f, y, nk, ncol, nk - 1)
    da, db, dc, df = (torch_dev(v) for v in (a, b, c, f))
    dx = torch.zeros((ncol, nk), dtype=torch.float64, device="cuda")
    pkg.tgx.trsolv_dev_mixed(da, db, dc, df, dx, 0, nk - 2, nsweep=nsweep)
    torch.cuda.synchronize()
    err = np.abs(dx.cpu().numpy()[:, :nk - 1] - y[:, :nk - 1]) / np.abs(y[:, :nk - 1])
    assert err.max() <= tol, err.max()


def test_dev_blktri2_blktri3_match_dropin(pkg, oracle):
    import torch
    from test_oracle_solvers import random_blocks, to_colmajor
    rng = np.random.default_rng(13)
    ncol, nk = 1000, 29
    for m, fn, ofn in ((2, pkg.tgx.blktri2_dev, None), (3, pkg.tgx.blktri3_dev, None)):
        P, Q, R, F = random_blocks(rng, ncol, nk, m)
        args = [to_colmajor(P), to_colmajor(Q), to_colmajor(R), np.ascontiguousarray(F)]
        y = np.zeros((ncol, nk, m))
        if m == 2:
            oracle.blktri(*args, y, 1, nk, 5, 5 + ncol - 1, 100000)
        else:
            oracle.blktri3(*args, y, nk, ncol, nk - 1)
        dx = torch.zeros((ncol, nk, m), dtype=torch.float64, device="cuda")
        fn(*[torch_dev(v) for v in args], dx, nk - 1)
        torch.cuda.synchronize()
        assert relerr(dx.cpu().numpy()[:, :nk - 1], y[:, :nk - 1]) <= 1e-14


def test_error_paths_do_not_abort(pkg):
    import torch
    t = torch.zeros((4, 10), dtype=torch.float64, device="cuda")
    with pytest.raises(pkg.tgx.TgxError):
        pkg.tgx.trsolv_dev(t, t, t, t, t, 0, 12)          # k2 beyond the column
    with pytest.raises(pkg.tgx.TgxError):
        pkg.tgx.trsolv_dev_mixed(t, t, t, t, t, 0, 5, nsweep=99)
    # zero columns is a no-op
    pkg.tgx.trsolv_dev(t, t, t, t, t, 0, 5, ncol=0)
    # drop-in with bad bounds reports through tgx_last_error
    a = np.zeros((3, 5))
    with pytest.raises(pkg.tgx.TgxError):
        pkg.tgx.trsolv(a, a, a, a, a.copy(), 1, 5, 0, 9, 1, 3, 3)


def test_solvers_from_two_host_threads_and_two_streams(pkg):
    """Thomas and block solves (both use library scratch) queued from two host
    threads at once, and from one thread on two streams without a wait in
    between, give bitwise the results of the same solves run one by one."""
    import threading
    import torch
    from test_oracle_solvers import random_blocks, to_colmajor
    rng = np.random.default_rng(21)
    jobs = []
    for ncol, nk in ((6000, 113), (3000, 57)):
        a, b, c, f = config1_system(rng, ncol, nk)
        P, Q, R, F = random_blocks(rng, ncol // 4, 29, 3)
        jobs.append(([torch_dev(v) for v in (a, b, c, f)], nk,
                     [torch_dev(v) for v in (to_colmajor(P), to_colmajor(Q), to_colmajor(R),
                                             np.ascontiguousarray(F))], ncol // 4))

    def run(job, stream=None):
        (sys_, nk, blk, nb) = job
        x = torch.zeros(sys_[0].shape, dtype=torch.float64, device="cuda")
        y = torch.zeros((nb, 29, 3), dtype=torch.float64, device="cuda")
        for _ in range(3):
            pkg.tgx.trsolv_dev(*sys_, x, 0, nk - 2, scheme=1, stream=stream)
            pkg.tgx.blktri3_dev(*blk, y, 28, stream=stream)
        return x, y

    ref = [run(j) for j in jobs]
    torch.cuda.synchronize()

    out, errs = [None, None], []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                out[i] = run(jobs[i], stream=s.cuda_stream)
            s.synchronize()
        except Exception as e:  # reported in the main thread
            errs.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(s1):
        o1 = run(jobs[0], stream=s1.cuda_stream)
    with torch.cuda.stream(s2):
        o2 = run(jobs[1], stream=s2.cuda_stream)
    torch.cuda.synchronize()
    for got in (out, [o1, o2]):
        for (rx, ry), (gx, gy) in zip(ref, got):
            assert torch.equal(rx, gx) and torch.equal(ry, gy)


SEG_ROWS = (1, 2, 3, 31, 32, 33, 57, 64, 65, 112, 113, 128, 129, 255, 256, 257)


def _segment_solve(pkg, nblk, sys_, x, n, col0=0):
    if nblk == 1:
        return pkg.tgx.trsolv_dev(*sys_, x, 0, n - 1, scheme=2, col0=col0, ncol=x.shape[0] - col0)
    a, b, c, f = (v[col0:] for v in sys_)
    return (pkg.tgx.blktri2_dev if nblk == 2 else pkg.tgx.blktri3_dev)(a, b, c, f, x[col0:], n)


@pytest.mark.parametrize("nblk", [1, 2, 3])
def test_partitioned_solver_row_counts(pkg, oracle, nblk):
    """Row counts at every edge of the segment sizes, column counts that leave
    a wavefront's last columns empty, rows beyond n and the unused couplings
    NaN (neither may be read into the solution), columns before col0
    untouched.  Diagonally dominant rows: each of the few dozen operations
    behind an unknown is an ulp at most, inside the block solvers' 1e-14."""
    import torch
    from test_oracle_solvers import to_colmajor
    for n in SEG_ROWS:
        for ncol, col0 in ((1, 0), (37, 0), (70, 5)):
            rng = np.random.default_rng(1000 * n + ncol)
            nk = n + (n + ncol) % 3
            A = rng.uniform(-1, 1, (ncol, nk, nblk, nblk))
            C = rng.uniform(-1, 1, (ncol, nk, nblk, nblk))
            B = rng.uniform(-1, 1, (ncol, nk, nblk, nblk))
            dom = np.abs(A).sum((2, 3)) + np.abs(B).sum((2, 3)) + np.abs(C).sum((2, 3))
            B = B + np.eye(nblk) * (dom + rng.uniform(.1, 1., (ncol, nk)))[..., None, None]
            F = rng.normal(size=(ncol, nk, nblk))
            y = np.zeros((ncol, nk, nblk))
            A[:, 0] = 0.
            C[:, n - 1] = 0.
            if nblk == 1:
                oracle.trsolv_ng(A[..., 0, 0], B[..., 0, 0], C[..., 0, 0], F[..., 0], y[..., 0], nk, ncol, n)
            elif nblk == 2:
                # blktri solves rows lev0..lev1-1: one level more than the rows
                ext = [np.concatenate([v[:, :n], v[:, :1]], axis=1) for v in (A, B, C, F)]
                z = np.zeros((ncol, n + 1, 2))
                oracle.blktri(*[to_colmajor(v) for v in ext[:3]], np.ascontiguousarray(ext[3]), z, 1, n + 1, 5,
                              5 + ncol - 1, 100000)
                y[:, :n] = z[:, :n]
            else:
                oracle.blktri3(to_colmajor(A), to_colmajor(B), to_colmajor(C), np.ascontiguousarray(F), y, nk, ncol, n)
            for v in (A, B, C, F):
                v[:, n:] = np.nan
            A[:, 0] = np.nan if nblk < 3 else 0.
            C[:, n - 1] = np.nan if nblk < 3 else 0.
            sys_ = [torch_dev(to_colmajor(v) if nblk > 1 else v[..., 0, 0]) for v in (A, B, C)]
            sys_.append(torch_dev(F if nblk > 1 else F[..., 0]))
            x = torch.full(sys_[3].shape, -5.0, dtype=torch.float64, device="cuda")
            print("case nblk=%d n=%d ncol=%d col0=%d" % (nblk, n, ncol, col0), flush=True)
            _segment_solve(pkg, nblk, sys_, x, n, col0)
            got = x.cpu().numpy().reshape(ncol, nk, nblk)
            assert np.all(got[:, n:] == -5.0) and np.all(got[:col0] == -5.0)
            assert relerr(got[col0:, :n], y[col0:, :n]) <= 1e-14, (n, ncol)


@pytest.mark.parametrize("nblk", [1, 2, 3])
@pytest.mark.parametrize("n", [24, 56, 112, 200])
def test_partitioned_solver_bad_segments(pkg, nblk, n):
    """Zero diagonal blocks where a segment starts: unsolvable segment by
    segment, well conditioned as a whole and for Thomas.  The other columns of
    the wavefront hold ordinary rows, one of them a NaN, which stays in its
    column.  Against a dense solve; the pattern (4, ..., 4, 0) with unit
    couplings has a condition number below 100, so 1e-12."""
    import torch
    ncol = 9
    eye = np.eye(nblk)
    B = np.tile(4. * eye, (ncol, n, 1, 1))
    A = np.tile(eye, (ncol, n, 1, 1))
    C = np.tile(eye, (ncol, n, 1, 1))
    rng = np.random.default_rng(n + nblk)
    F = rng.normal(size=(ncol, n, nblk))
    B[2::3, 8::8] = 0.        # a multiple of every segment length
    F[4, n // 2, 0] = np.nan
    A[:, 0] = 0.
    C[:, n - 1] = 0.
    sys_ = [torch_dev(v if nblk > 1 else v[..., 0, 0]) for v in (A, B, C)] + [torch_dev(F if nblk > 1 else F[..., 0])]
    x = torch.zeros(sys_[3].shape, dtype=torch.float64, device="cuda")
    _segment_solve(pkg, nblk, sys_, x, n)
    got = x.cpu().numpy().reshape(ncol, n, nblk)
    assert np.isnan(got[4]).any()
    for col in range(ncol):
        if col == 4:
            continue
        M = np.zeros((n * nblk, n * nblk))
        for k in range(n):
            s = slice(k * nblk, (k + 1) * nblk)
            M[s, s] = B[col, k]
            if k:
                M[s, (k - 1) * nblk:k * nblk] = A[col, k]
            if k < n - 1:
                M[s, (k + 1) * nblk:(k + 2) * nblk] = C[col, k]
        assert np.linalg.cond(M) < 100.
        ref = np.linalg.solve(M, F[col].ravel()).reshape(n, nblk)
        assert relerr(got[col], ref) <= 1e-12, (col, relerr(got[col], ref))
    if nblk == 1:  # solved again in the reference's order: bit for bit the Thomas scheme
        y = torch.zeros_like(x)
        pkg.tgx.trsolv_dev(*sys_, y, 0, n - 1, scheme=1)
        assert torch.equal(x[2::3], y[2::3])


@pytest.mark.parametrize("n", [1, 2, 3, 57, 63, 64, 65, 95, 96, 128, 255, 256, 511, 512])
def test_thomas_scheme_bit_for_bit(pkg, n):
    """The Thomas scheme in the reference's order, trsolv.F:38-54, exactly: rows
    at the limits of each LDS form and beyond (512), blocks with and without
    columns left over, columns from the middle of the batch, rows from the middle
    of the levels; nothing else of x is written, and what no equation reads (NaN
    here) does not enter."""
    import torch
    rng = np.random.default_rng(n)
    for ncol, col0, k1, pad in ((1, 0, 0, 0), (7, 3, 1, 2), (16, 0, 0, 1), (33, 5, 2, 0)):
        ldk = k1 + n + pad
        tot = col0 + ncol + 2
        a, c = -rng.uniform(.5, 2., (tot, ldk)), -rng.uniform(.5, 2., (tot, ldk))
        b = -(a + c) + rng.uniform(.1, 1., (tot, ldk))
        f = rng.normal(0., 5., (tot, ldk))
        k2 = k1 + n - 1
        a[:, k1] = np.nan
        c[:, k2] = np.nan
        x = np.full((tot, ldk), -7.)
        ref = x.copy()
        cols = slice(col0, col0 + ncol)
        w1, w3 = b[cols, k1], f[cols, k1] / b[cols, k1]
        ref[cols, k1] = w3
        w2s = np.zeros((ncol, ldk))
        for k in range(k1 + 1, k2 + 1):
            w2 = c[cols, k - 1] / w1
            w2s[:, k - 1] = w2
            w1 = b[cols, k] - a[cols, k] * w2
            w3 = (f[cols, k] - a[cols, k] * w3) / w1
            ref[cols, k] = w3
        for k in range(k2 - 1, k1 - 1, -1):
            ref[cols, k] = ref[cols, k] - w2s[:, k] * ref[cols, k + 1]
        d = [torch_dev(v) for v in (a, b, c, f, x)]
        print("case", n, ncol, flush=True)
        pkg.tgx.trsolv_dev(*d, k1, k2, scheme=pkg.tgx.SCHEME_THOMAS, col0=col0, ncol=ncol)
        torch.cuda.synchronize()
        assert np.array_equal(d[4].cpu().numpy(), ref), (n, ncol)


def _growing_segments(nblk, n, period, g, ncol, seed):
    """Columns whose rows taken `period` at a time grow by about g per row of a
    segment, although the whole column is well conditioned (and Thomas, which
    never meets the small pivots unreduced, solves it to rounding): segment
    starts 1/g between unit couplings, rows inside 1 + 1/g after a coupling 1/g,
    the last row 2.5.  Rows, and the condition number of the scalar column."""
    k = np.arange(n)
    e = k % period
    b = np.where(k == 0, 2., np.where(e == 0, 1. / g, np.where(e == period - 1, 2.5, 1. + 1. / g)))
    a = np.where((e == 0) | (e == period - 1), 1., 1. / g)
    eye = np.eye(nblk)
    A, B = (np.tile(v[:, None, None] * eye, (ncol, 1, 1, 1)) for v in (a, b))
    C = np.tile(eye, (ncol, n, 1, 1))
    F = np.random.default_rng(seed).normal(size=(ncol, n, nblk))
    A[:, 0] = 0.
    C[:, n - 1] = 0.
    return A, B, C, F, np.linalg.cond(np.diag(b) + np.diag(a[1:], -1) + np.diag(np.ones(n - 1), 1))


def _device_segments(pkg, nblk, A, B, C, F):
    import torch
    from test_oracle_solvers import to_colmajor
    sys_ = [torch_dev(to_colmajor(v) if nblk > 1 else v[..., 0, 0]) for v in (A, B, C)]
    sys_.append(torch_dev(F if nblk > 1 else F[..., 0]))
    x = torch.zeros_like(sys_[3])
    _segment_solve(pkg, nblk, sys_, x, F.shape[1])
    return x.cpu().numpy().reshape(F.shape)


def _refined(A, B, C, F):
    """The solutions of block tridiagonal columns, refined to beyond 64 bits."""
    ncol, n, m = F.shape
    M = np.zeros((ncol, n, m, n, m))
    for k in range(n):
        M[:, k, :, k] = B[:, k]
        if k:
            M[:, k, :, k - 1] = A[:, k]
        if k < n - 1:
            M[:, k, :, k + 1] = C[:, k]
    M = M.reshape(ncol, n * m, n * m)
    f = F.reshape(ncol, n * m, 1)
    x = np.linalg.solve(M, f).astype(np.longdouble)
    for _ in range(3):
        r = f - np.stack([(Mi.astype(np.longdouble) @ xi) for Mi, xi in zip(M, x)])
        x = x + np.linalg.solve(M, r.astype(np.float64))
    return x.reshape(F.shape)


@pytest.mark.parametrize("nblk", [2, 3])
@pytest.mark.parametrize("n", [56, 112, 200])
def test_block_rows_with_a_large_correction(pkg, nblk, n):
    """A block column whose correction from the residual shows that its
    segments lost digits is not stored: an accepted correction is at most 1e-12
    of the unknowns and all that an error contracts by is the unit couplings
    over 2.5 (a factor of 5 at most), so 5e-12."""
    A, B, C, F, cond = _growing_segments(nblk, n, 4, 31., 40, n + nblk)
    assert cond < 400.
    assert relerr(_device_segments(pkg, nblk, A, B, C, F), _refined(A, B, C, F).astype(np.float64)) <= 5e-12


@pytest.mark.parametrize("nblk", [1, 2, 3])
@pytest.mark.parametrize("n", [28, 56, 112, 200])
def test_partitioned_solver_growing_segments(pkg, oracle, nblk, n):
    """Columns whose multipliers compound over a segment, for segments of 2, 4
    and 8 rows, one small pivot per segment on its own, multipliers on both
    sides of every limit the kernel could put to a single one.  Accepted columns
    have multipliers and products of them of at most 4 and the others are solved
    in the reference's order, so the worst error stays within twice that (a
    substitution and a reduction use them) of the reference order's."""
    from test_oracle_solvers import to_colmajor
    parts, what = [], []
    for g in (2.2, 5., 10., 20., 31., 33.):
        for period in (2, 4, 8):
            *p, cond = _growing_segments(nblk, n, period, g, 4, int(100 * g) + period)
            if cond < 400.:
                parts.append(p)
                what += [(g, period)] * 4
            k = np.arange(n)
            A, _, C, F = (v.copy() for v in p)
            A[:, 1:] = C[:, :n - 1] = np.eye(nblk)
            B = np.tile(np.where((k % period == 0) & (k > 0), 1. / g, 4.)[:, None, None] * np.eye(nblk), (4, 1, 1, 1))
            if period > 2:
                parts.append([A, B, C, F])
                what += [(g, -period)] * 4
    A, B, C, F = (np.concatenate(v) for v in zip(*parts))
    ncol = len(what)
    y = np.zeros_like(F)
    if nblk == 1:
        oracle.trsolv_ng(*(np.ascontiguousarray(v[..., 0, 0]) for v in (A, B, C)), np.ascontiguousarray(F[..., 0]),
                         y[..., 0], n, ncol, n)
    elif nblk == 2:
        ext = [np.concatenate([v, v[:, :1]], axis=1) for v in (A, B, C, F)]
        z = np.zeros((ncol, n + 1, 2))
        oracle.blktri(*[to_colmajor(v) for v in ext[:3]], np.ascontiguousarray(ext[3]), z, 1, n + 1, 5, 5 + ncol - 1, 100000)
        y = z[:, :n]
    else:
        oracle.blktri3(to_colmajor(A), to_colmajor(B), to_colmajor(C), F, y, n, ncol, n)
    exact = _refined(A, B, C, F)
    scale = np.abs(exact).max(axis=(1, 2))
    err = [(np.abs(v - exact).max(axis=(1, 2)) / scale).astype(np.float64) for v in (_device_segments(pkg, nblk, A, B, C, F), y)]
    worst = int(np.argmax(err[0]))
    assert err[0].max() <= 8. * err[1].max(), (what[worst], err[0].max(), err[1].max())


@pytest.mark.parametrize("n", [56, 65, 112, 128, 200, 256])
def test_partitioned_solver_slowly_refined_columns(pkg, oracle, n):
    """One pivot of 1e-2.5 to 1 in eight rows: multipliers compound to 1e10 and
    more, so that a correction tells little of the next.  The last one is within
    1e-13 of the unknowns, and what the reference's order solves has its error."""
    k, nc = np.arange(n) % 8, 256
    g = np.logspace(0., 2.5, nc)[:, None]
    A = np.where((k == 0) | (k == 7), 1., 1. / g)
    B = np.where(k == 0, 1. / g, np.where(k == 7, 2.5, 1. + 1. / g))
    C, F = np.ones((nc, n)), np.random.default_rng(n).standard_normal((nc, n))
    B[:, 0] = 2.
    A[:, 0] = C[:, -1] = 0.
    A, B, C, F = (v.reshape(nc, n, 1, 1) for v in (A, B, C, F))
    F = F[..., 0]
    exact = _refined(A, B, C, F)
    scale = np.abs(exact).max(axis=(1, 2))
    y = np.zeros((nc, n))
    oracle.trsolv_ng(*(np.ascontiguousarray(v[..., 0, 0]) for v in (A, B, C)), np.ascontiguousarray(F[..., 0]), y, n, nc, n)
    err = [(np.abs(v - exact).max(axis=(1, 2)) / scale).astype(np.float64)
           for v in (_device_segments(pkg, 1, A, B, C, F), y[..., None])]
    assert err[0].max() <= 1e-13 + err[1].max(), (g[int(np.argmax(err[0])), 0], err[0].max(), err[1].max())


@pytest.mark.parametrize("nblk", [1, 2, 3])
@pytest.mark.parametrize("n", [28, 56, 112, 200])
def test_partitioned_solver_in_place(pkg, nblk, n):
    """The solution written over the right-hand side: columns that are refined
    read theirs again after their neighbours in the wavefront have been stored."""
    import torch
    from test_oracle_solvers import to_colmajor
    parts = [_growing_segments(nblk, n, period, g, 3, n + period)[:4] for g in (1., 31.) for period in (4, 8)]
    A, B, C, F = (np.concatenate(v) for v in zip(*parts))
    B[1::4, ::8] = 0.  # and in the reference's order
    B[:, 0] = 2. * np.eye(nblk)
    perm = np.random.default_rng(n).permutation(len(F))
    A, B, C, F = (v[perm] for v in (A, B, C, F))
    sys_ = [torch_dev(to_colmajor(v) if nblk > 1 else v[..., 0, 0]) for v in (A, B, C)]
    sys_.append(torch_dev(F if nblk > 1 else F[..., 0]))
    x = torch.zeros_like(sys_[3])
    _segment_solve(pkg, nblk, sys_, x, n)
    _segment_solve(pkg, nblk, sys_, sys_[3], n)
    assert torch.equal(x, sys_[3]) and bool(torch.isfinite(x).all())


@pytest.mark.parametrize("nblk", [2, 3])
@pytest.mark.parametrize("n", [1, 2, 57, 256, 257])
def test_block_rows_in_the_reference_order(pkg, oracle, nblk, n):
    """TGX_SCHEME_THOMAS on block rows: the oracle's order of operations, to its
    own 1e-14 on dominant rows, also where the default takes another (2 to 256
    rows, whose bits differ); an unknown scheme is refused."""
    import torch
    from test_oracle_solvers import to_colmajor
    rng = np.random.default_rng(n)
    ncol = 70
    A, B, C = (rng.uniform(-1, 1, (ncol, n, nblk, nblk)) for _ in range(3))
    B = B + np.eye(nblk) * (np.abs(A) + np.abs(B) + np.abs(C)).sum((2, 3), keepdims=True)
    F = rng.normal(size=(ncol, n, nblk))
    A[:, 0] = 0.
    C[:, n - 1] = 0.
    y = np.zeros_like(F)
    if nblk == 2:
        ext = [np.concatenate([v, v[:, :1]], axis=1) for v in (A, B, C, F)]
        z = np.zeros((ncol, n + 1, 2))
        oracle.blktri(*[to_colmajor(v) for v in ext[:3]], np.ascontiguousarray(ext[3]), z, 1, n + 1, 5, 5 + ncol - 1, 100000)
        y = z[:, :n]
    else:
        oracle.blktri3(to_colmajor(A), to_colmajor(B), to_colmajor(C), F, y, n, ncol, n)
    solve = pkg.tgx.blktri2_dev if nblk == 2 else pkg.tgx.blktri3_dev
    sys_ = [torch_dev(to_colmajor(v)) for v in (A, B, C)] + [torch_dev(F)]
    x, d = (torch.zeros_like(sys_[3]) for _ in range(2))
    solve(*sys_, x, n, scheme=pkg.tgx.SCHEME_THOMAS)
    assert relerr(x.cpu().numpy(), y) <= 1e-14
    solve(*sys_, d, n)
    assert torch.equal(x, d) == (n > 256) or n == 1
    with pytest.raises(pkg.tgx.TgxError):
        solve(*sys_, x, n, scheme=7)
