"""The Krylov loops inside one resident grid (neon_amd/csrc/grid_kernels.hpp) at the sizes where
their layouts can go wrong, against the launch-per-phase loops (which a solve takes while kernel
timing is on) and the true residual of the downloaded or host matrix.

Tolerances: both loops stop on a recurrence residual of 1e-10 |b|; the true residual differs from
it by the rounding of the recurrence, some eps |A| |x| per iteration, below 1e-11 |b| on these
systems (condition below 1e5), so it is held to 1.1e-10 |b|.  The iteration counts differ only where
the last residual lands within rounding of the tolerance: 2 or 2 %, as for the oracle's counts."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse.linalg
import scipy.sparse as sp

import neon_amd
from neon_amd import _capi, problems

pytestmark = pytest.mark.gpu


def _both(ctx, solve):
    """solve() on the resident grid and by launches."""
    grid = solve()
    ctx.profile(True)
    try:
        launches = solve()
    finally:
        ctx.profile(False)
    return grid, launches


def _check(A, b, grid, launches):
    for x, its, _ in (grid, launches):
        res = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
        assert res <= 1.1e-10, res
    assert abs(grid[1] - launches[1]) <= max(2, 0.02 * launches[1]), (grid[1], launches[1])


# One to three slices; the last with one node; eight wavefronts per slice with two and four items
# each; four per slice; several rounds; one wavefront per slice; two rounds of it; and the rows too
# many for every vector to stay in LDS.  The plates' slices have up to 31 entries, the generated
# numbering none of the common offsets (the full copy).
MESHES = [((1, 1, 1), "grid", 0.0), ((3, 3, 3), "grid", 0.0), ((4, 4, 4), "grid", 0.0), ((12, 4, 4), "grid", 0.0),
          ((20, 21, 19), "grid", 0.0), ((29, 31, 30), "grid", 0.0), ((35, 33, 34), "grid", 0.0),
          ((43, 40, 41), "grid", 0.0), ((52, 50, 51), "grid", 0.0), ((66, 65, 64), "grid", 0.0),
          ((24, 12, 6), "grid", 1.5), ((64, 32, 20), "grid", 4.0),
          ((5, 4, 6), "shuffled", 0.0), ((23, 22, 24), "shuffled", 0.0), ((31, 30, 33), "boundary", 0.0),
          ((45, 44, 46), "boundary", 0.0)]


def _mesh(ctx, dims, numbering, hole):
    if hole:
        p = problems.notched_plate_j2(*dims, hole_cells=hole)
        model = neon_amd.MODEL_LINEAR_ELASTIC
    else:
        p = problems.block_rollers(max(dims), dims=dims)
        model = p.model
    X, conn, ijk, fixed = p.X, p.conn, p.ijk, p.fixed_dofs()
    if numbering != "grid":
        if numbering == "shuffled":
            order = np.random.default_rng(3).permutation(len(X))
        else:
            faces = np.sum((ijk == 0) | (ijk == np.array(dims)), axis=1)
            order = np.argsort(-faces, kind="stable")
        new = np.empty(len(order), np.int32)
        new[order] = np.arange(len(order), dtype=np.int32)
        X, conn = X[order], new[conn]
        fixed = np.sort(3 * new[fixed // 3] + fixed % 3).astype(np.int32)
    mg = neon_amd.DeviceMesh(X, conn, p.params, model=model, context=ctx)
    mg.update_internal_variables()
    mg.assemble()
    b = np.random.default_rng(11).standard_normal(mg.n_dofs)
    mg.enforce_dirichlet(fixed, b)
    return mg, b


def _matrix(mg):
    rp, ci = mg.pattern()
    val, _ = mg.download(internal_force=False)
    return sp.csr_matrix((val, ci, rp))


@pytest.mark.parametrize("dims,numbering,hole", MESHES)
def test_cg_on_the_mesh_tangent(ctx, dims, numbering, hole):
    print(dims, numbering, hole, flush=True)
    mg, b = _mesh(ctx, dims, numbering, hole)
    grid, launches = _both(ctx, lambda: mg.solve(b, tol=1e-10))
    _check(_matrix(mg), b, grid, launches)


def test_cg_with_32bit_offsets(ctx):
    mg, b = _mesh(ctx, (12, 11, 13), "shuffled", 0.0)
    mg.spmv_config(flags=neon_amd.SPMV_SLICED | neon_amd.SPMV_INDEX32)
    grid, launches = _both(ctx, lambda: mg.solve(b, tol=1e-10))
    _check(_matrix(mg), b, grid, launches)


def _spd(n, per_row, seed, long_rows=0):
    """A diagonally dominant symmetric matrix of n rows with about per_row entries each, every
    seventh row its diagonal alone, and long_rows rows that couple to every row."""
    rng = np.random.default_rng(seed)
    m = n * per_row // 2
    i, j = rng.integers(0, n, m), rng.integers(0, n, m)
    keep = (i % 7 != 0) & (j % 7 != 0) & (i != j)
    i, j = i[keep], j[keep]
    for r in range(long_rows):
        i = np.concatenate([i, np.full(n - 1, n // 2 + r)])
        j = np.concatenate([j, np.delete(np.arange(n), n // 2 + r)])
    S = sp.coo_matrix((rng.uniform(-1, 1, len(i)), (i, j)), shape=(n, n)).tocsr()
    S = S + S.T
    S = (S + sp.diags(np.abs(S).sum(axis=1).A1 * 1.05 + 1.0)).tocsr()
    S.sort_indices()
    return S, rng.standard_normal(n)


# one row; a block's 64 rows and one more; chunks of 4,096 entries with rows across their ends;
# rows longer than a chunk; many blocks, all vectors in LDS and not
CSR = [(1, 1, 0), (15, 3, 0), (64, 5, 0), (65, 5, 0), (1000, 90, 0), (6000, 12, 2), (16384, 6, 0), (70001, 30, 0),
       (300007, 8, 0), (1200000, 4, 0)]


def _solve_csr(ctx, cls, A, b, tol=1e-10, criterion=neon_amd.STOP_RELATIVE):
    s = cls(tol, 4000, criterion=criterion, context=ctx)
    x = np.zeros(len(b))
    s.solve(A, x, b)
    return x, s.iterations, s.error


@pytest.mark.parametrize("n,per_row,long_rows", CSR)
def test_cg_on_host_csr(ctx, n, per_row, long_rows):
    print(n, per_row, long_rows, flush=True)
    A, b = _spd(n, per_row, n, long_rows)
    grid, launches = _both(ctx, lambda: _solve_csr(ctx, neon_amd.conjugate_gradient_hip, A, b))
    _check(A, b, grid, launches)


def _with_rows(n, lengths, seed):
    """Diagonally dominant, symmetric: the first rows have these lengths (diagonal included), over the
    columns after theirs; the others the diagonal, their parts of those and a neighbour."""
    rng = np.random.default_rng(seed)
    i = np.concatenate([np.full(k - 1, r) for r, k in enumerate(lengths)])
    m = len(lengths)
    j = np.concatenate([np.sort(rng.choice(np.arange(m, n), k - 1, replace=False)) for k in lengths])
    far = np.arange(m, n - 1)
    i, j = np.concatenate([i, far]), np.concatenate([j, far + 1])
    S = sp.coo_matrix((rng.uniform(-1, 1, len(i)), (i, j)), shape=(n, n)).tocsr()
    S = S + S.T
    S = (S + sp.diags(np.abs(S).sum(axis=1).A1 * 1.05 + 1.0)).tocsr()
    S.sort_indices()
    assert list(np.diff(S.indptr)[:m]) == list(lengths)
    return S, rng.standard_normal(n)


# Rows at the length from which a wavefront adds them up (256 entries of a chunk), in one workgroup and
# in several; a chunk full of such rows; rows of a chunk and more; and rows so unequal that the launch
# loop takes the system
@pytest.mark.parametrize("n,lengths", [(600, [255, 256, 257, 258]), (5000, [255, 256, 257, 258, 512]),
                                       (5000, [257] * 40), (40000, [4095, 4096, 4097, 9000]), (70000, [300] * 64),
                                       (30000, [20000] * 64)])
def test_cg_and_bicgstab_on_long_rows(ctx, n, lengths):
    print(n, len(lengths), flush=True)
    A, b = _with_rows(n, lengths, n)
    for cls in (neon_amd.conjugate_gradient_hip, neon_amd.biconjugate_gradient_stabilised_hip):
        grid, launches = _both(ctx, lambda: _solve_csr(ctx, cls, A, b))
        for x, its, _ in (grid, launches):
            assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)
        assert abs(grid[1] - launches[1]) <= 3 + 0.15 * launches[1], (grid[1], launches[1])


def test_unequal_rows_cost_no_more_than_the_launch_loop(ctx):
    """64 full rows of 20,000: the solve must not be far slower than the launch loop (it was 13 times).
    The least of three calls each; 2 for the scatter (the launch loop's calls are timed per kernel)."""
    import time

    A, b = _with_rows(20064, [20000] * 64, 3)
    arrays = (A.indptr, A.indices, A.data)

    def timed():
        times = []
        for _ in range(3):
            start = time.perf_counter()
            _solve_csr(ctx, neon_amd.conjugate_gradient_hip, arrays, b)
            times.append(time.perf_counter() - start)
        return min(times)

    timed()
    grid, launches = _both(ctx, timed)
    print(grid, launches, flush=True)
    assert grid <= 2.0 * launches


def _chain(n, shift):
    return sp.diags([-np.ones(n - 1), np.full(n, 2.0 + shift), -np.ones(n - 1)], [-1, 0, 1], format="csr")


def _laplacian(m):
    one = sp.identity(m)
    return sp.csr_matrix(sp.kron(_chain(m, 0.0), one) + sp.kron(one, _chain(m, 0.0)))


# Systems of one workgroup (at most 1,024 rows and 8,192 entries) whose solves take several launches
# of 64 iterations: a continued launch gathers p from LDS, which it has filled from global memory.
ONE_WORKGROUP = {"laplacian 30x30": lambda: _laplacian(30), "chain 1000": lambda: _chain(1000, 0.01),
                 "chain 1024": lambda: _chain(1024, 0.01), "chain 65": lambda: _chain(65, 1e-4)}


@pytest.mark.parametrize("name", ONE_WORKGROUP)
def test_cg_of_one_workgroup_over_several_launches(ctx, name):
    """The true residual differs from the recurrence's by at most eps |A| |x| per iteration (|A| <= 8);
    each solve repeats bit for bit."""
    print(name, flush=True)
    A = ONE_WORKGROUP[name]()
    b = np.random.default_rng(13).standard_normal(A.shape[0])
    grid, launches = _both(ctx, lambda: _solve_csr(ctx, neon_amd.conjugate_gradient_hip, A, b))
    assert grid[1] > 64 or name == "chain 65"
    for x, its, _ in (grid, launches):
        drift = its * np.finfo(float).eps * 8.0 * np.linalg.norm(x)
        assert np.linalg.norm(b - A @ x) <= 1e-10 * np.linalg.norm(b) + drift
    assert abs(grid[1] - launches[1]) <= max(2, 0.02 * launches[1]), (grid[1], launches[1])
    # other systems of one workgroup on the same compute units' LDS in between
    for k in range(3):
        other, c = _spd(700 + k, 5, 40 + k)
        _solve_csr(ctx, neon_amd.conjugate_gradient_hip, other, c)
        again = _solve_csr(ctx, neon_amd.conjugate_gradient_hip, A, b)
        assert np.array_equal(again[0], grid[0]) and again[1] == grid[1]


@pytest.mark.parametrize("limit", [64, 65, 129])
def test_cg_of_one_workgroup_stops_at_the_limit(ctx, limit):
    """The limit at the end of a launch, and after the first iteration of the second and of the third
    one.  The iterate that is left meets the a-priori bound of k conjugate gradient iterations,
    |x_k - x|_A <= 2 ((sqrt(c) - 1) / (sqrt(c) + 1))^k |x|_A (the Jacobi scaling is by one number, and
    c < 4.01 / 0.01 for this chain)."""
    A = _chain(1000, 0.01)
    b = np.random.default_rng(14).standard_normal(1000)
    exact = scipy.sparse.linalg.spsolve(A.tocsc(), b)
    rate = (np.sqrt(401.0) - 1.0) / (np.sqrt(401.0) + 1.0)
    for timed in (False, True):
        s = neon_amd.conjugate_gradient_hip(1e-30, limit, criterion=neon_amd.STOP_RELATIVE, context=ctx)
        x = np.zeros(1000)
        ctx.profile(timed)
        try:
            with pytest.raises(neon_amd.computational_error) as e:
                s.solve(A, x, b)
        finally:
            ctx.profile(False)
        assert (e.value.code, s.iterations) == (_capi.NEON_NONCONVERGED, limit)
        d = x - exact
        assert np.sqrt(d @ (A @ d)) <= 2.0 * rate ** limit * np.sqrt(exact @ b)


@pytest.mark.parametrize("criterion", [neon_amd.STOP_RELATIVE, neon_amd.STOP_ABSOLUTE_PRECONDITIONED])
def test_cg_ends(ctx, criterion):
    """A zero right-hand side, the iteration limit inside and at the end of a launch, and values
    that are not finite end as they do by launches."""
    mg, b = _mesh(ctx, (12, 4, 4), "grid", 0.0)
    solve = dict(criterion=criterion, tol=1e-30)
    x, its, err = mg.solve(np.zeros_like(b), **solve)
    assert its == 0 and err == 0.0 and not x.any()
    A = _matrix(mg)
    for limit in (1, 63, 64, 65):
        outcomes = []
        for timed in (False, True):
            s = neon_amd.conjugate_gradient_hip(1e-30, limit, criterion=criterion, context=ctx)
            x = np.zeros_like(b)
            ctx.profile(timed)
            try:
                with pytest.raises(neon_amd.computational_error) as e:
                    s.solve(A, x, b)
            finally:
                ctx.profile(False)
            outcomes.append((e.value.code, s.iterations))
        assert outcomes == [(_capi.NEON_NONCONVERGED, limit)] * 2
    b[17] = np.inf
    with pytest.raises(neon_amd.computational_error) as e:
        mg.solve(b, **solve)
    assert e.value.code == _capi.NEON_NAN_OR_INF


def test_a_grid_that_gives_up_is_solved_by_launches(ctx):
    """With no patience the first wait of a workgroup for another ends the grid, and then the one-launch
    vector part of the launch loop; the solve takes separate launches, and the next one with
    patience the grid again.  The same for the mixed loop."""
    fn = _capi.measure_lib().neon_test_grid_patience
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_int64]
    A, b = _spd(40000, 20, 8)

    def solve():
        return _solve_csr(ctx, neon_amd.conjugate_gradient_hip, A, b)

    mg, bm = _mesh(ctx, (30, 29, 31), "grid", 0.0)
    mg.assemble(neon_amd.PRECISION_MIXED)
    mg.enforce_dirichlet(problems.block_rollers(31, dims=(30, 29, 31)).fixed_dofs(), bm)

    def mixed():
        return mg.solve(bm, tol=1e-10)

    grid, launches = _both(ctx, solve)
    patient = mixed()
    ctx.check(fn(ctx.handle, 0))
    try:
        impatient, impatient_mixed = solve(), mixed()
    finally:
        ctx.check(fn(ctx.handle, 10 ** 8))
    _check(A, b, impatient, launches)
    _check(_matrix(mg), bm, impatient_mixed, patient)
    again = solve()
    assert np.array_equal(again[0], grid[0]) and again[1] == grid[1]
    assert np.array_equal(mixed()[0], patient[0])


def test_a_grid_that_gave_up_rests(ctx):
    """After a grid has given up, the context's solves take launches for a while (64 times what was
    lost, at least 0.64 s) instead of each waiting again; then the grid is tried once more.  With
    no patience every try gives up, so the count of give-ups is the count of tries.  A solve whose
    grid gave up does not try the one-launch vector part either; the vector part of a system too
    large for the grid, and of the mixed loop, gives up as the grid does."""
    import time

    lib = _capi.measure_lib()
    patience, count = lib.neon_test_grid_patience, lib.neon_test_grid_give_ups
    patience.restype, patience.argtypes = C.c_int, [C.c_void_p, C.c_int64]
    count.restype, count.argtypes = C.c_int, [C.c_void_p, C.POINTER(C.c_int64)]

    def tries():
        n = C.c_int64(0)
        ctx.check(count(ctx.handle, C.byref(n)))
        return n.value

    A, b = _spd(40000, 20, 8)
    big, bb = _spd(1300000, 4, 9)
    mg, bm = _mesh(ctx, (30, 29, 31), "grid", 0.0)
    mg.assemble(neon_amd.PRECISION_MIXED)
    mg.enforce_dirichlet(problems.block_rollers(31, dims=(30, 29, 31)).fixed_dofs(), bm)
    solve = lambda: _solve_csr(ctx, neon_amd.conjugate_gradient_hip, A, b)
    solves = [lambda: _solve_csr(ctx, neon_amd.conjugate_gradient_hip, big, bb), lambda: mg.solve(bm, tol=1e-10)]
    solve()  # the memory the context keeps
    try:
        ctx.check(patience(ctx.handle, 0))
        start, first = time.perf_counter(), tries()
        x = solve()[0]
        done = 1
        while time.perf_counter() - start < 0.3:
            assert np.array_equal(solve()[0], x)
            done += 1
        assert done >= 5 and tries() == first + 1, (done, tries() - first)
        time.sleep(1.0)
        # the try before took less than 10 ms of waiting and work, or 64 times that is over by now
        assert np.array_equal(solve()[0], x)
        assert tries() <= first + 2
        for other in solves:
            ctx.check(patience(ctx.handle, 0))  # ends the rest
            n = tries()
            other()
            assert tries() == n + 1
            other()
            assert tries() == n + 1
    finally:
        ctx.check(patience(ctx.handle, 10 ** 8))
    assert np.linalg.norm(b - A @ x) <= 1.1e-10 * np.linalg.norm(b)


# numbers left for a first launch and not for the second; and for none
@pytest.mark.parametrize("left", [300, 1])
def test_the_exchange_numbers_start_again(left):
    """A context's exchanges are numbered in 32 bits.  Where the numbers run out the slots are cleared
    and the numbers start again at 1, in the middle of a solve too: every result has the bits it
    has on a fresh context, CG (grid, small grid and the launch loop's vector part) and BiCGSTAB."""
    set_number = _capi.measure_lib().neon_test_grid_epoch
    set_number.restype, set_number.argtypes = C.c_int, [C.c_void_p, C.c_uint32]
    A, b = _spd(40000, 20, 8)
    U, ub = _unsymmetric(20000, 30, 6)
    lap = _laplacian(120)
    cg, bi = neon_amd.conjugate_gradient_hip, neon_amd.biconjugate_gradient_stabilised_hip
    out = {}
    for key in ("fresh", "wrapped"):
        c = neon_amd.Context(0)
        try:
            mg, bm = _mesh(c, (20, 21, 19), "grid", 0.0)
            solves = [lambda: _solve_csr(c, cg, A, b), lambda: _solve_csr(c, cg, lap, np.ones(14400)),
                      lambda: _solve_csr(c, bi, U, ub), lambda: mg.solve(bm, tol=1e-10)]
            results = []
            for solve in solves:
                if key == "wrapped":
                    c.check(set_number(c.handle, 2 ** 32 - 1 - left))
                results.append(solve())
            mg.assemble(neon_amd.PRECISION_MIXED)
            mg.enforce_dirichlet(problems.block_rollers(21, dims=(20, 21, 19)).fixed_dofs(), bm.copy())
            if key == "wrapped":
                c.check(set_number(c.handle, 2 ** 32 - 1 - min(left, 20)))
            results.append(mg.solve(bm, tol=1e-10))
            out[key] = results
            del mg
        finally:
            c.close()
    for fresh, wrapped in zip(out["fresh"], out["wrapped"]):
        assert np.array_equal(fresh[0], wrapped[0]) and fresh[1] == wrapped[1]


# one workgroup, its last entries fewer than a 16-byte group; several; and more entries than the
# threads keep in registers
@pytest.mark.parametrize("dims", [(1, 1, 1), (7, 6, 5), (20, 19, 23), (44, 43, 45), (104, 102, 101)])
def test_mixed_cg_vector_part(ctx, dims):
    """The mixed loop's one-launch vector part: the true residual against the FP32 tangent, and the
    FP64 solve's iteration count (reliable updates keep the Krylov space: within 25 % and 8, the
    test's period)."""
    print(dims, flush=True)
    mg, b = _mesh(ctx, dims, "grid", 0.0)
    its64 = mg.solve(b, tol=1e-8)[1]
    p = problems.block_rollers(max(dims), dims=dims)
    mg.assemble(neon_amd.PRECISION_MIXED)
    mg.enforce_dirichlet(p.fixed_dofs(), b)
    x, its, _ = mg.solve(b, tol=1e-8)
    assert np.linalg.norm(b - _matrix(mg) @ x) <= 1.1e-8 * np.linalg.norm(b)
    assert its <= 1.25 * its64 + 8, (its, its64)


def test_a_small_full_copy_is_read_through_the_caches(ctx):
    """The mixed loop's FP32 product on a full copy of 3 MB (boundary-first numbering), right after the
    assembly: the default flags, which ask for nontemporal loads, must not make it slower than plain
    loads do (they did by 40 %).  Least of five alternating runs; 20 % for the scatter of runs.  The
    loads' kind does not change the solution."""
    mg, b = _mesh(ctx, (14, 14, 14), "boundary", 0.0)
    fixed = np.flatnonzero(b == 0.0).astype(np.int32)
    plain = neon_amd.SPMV_SLICED | neon_amd.SPMV_SYMMETRIC
    best, x = {}, {}
    for _ in range(5):
        for flags in (plain | neon_amd.SPMV_NONTEMPORAL, plain):
            mg.spmv_config(flags=flags)
            mg.assemble(neon_amd.PRECISION_MIXED)
            mg.enforce_dirichlet(fixed, b.copy())
            ctx.profile(True)
            try:
                x[flags] = mg.solve(b, tol=1e-10)[0]
                count, ms = ctx.profile_read(_capi.KERNEL_SPMV_FP32)
            finally:
                ctx.profile(False)
            best[flags] = min(best.get(flags, np.inf), ms / count)
    print(best, flush=True)
    assert np.array_equal(x[plain], x[plain | neon_amd.SPMV_NONTEMPORAL])
    assert best[plain | neon_amd.SPMV_NONTEMPORAL] <= 1.2 * best[plain]


def test_two_contexts_share_the_gpu():
    """Solves on two contexts from two threads at once: the grids take turns for the compute units."""
    import threading

    results = {}

    def work(k):
        c = neon_amd.Context(0)
        try:
            A, b = _spd(200000, 20, 30 + k)
            results[k] = [_solve_csr(c, neon_amd.conjugate_gradient_hip, A, b)[0] for _ in range(3)]
            results[k].append(np.linalg.norm(b - A @ results[k][0]) / np.linalg.norm(b))
        finally:
            c.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert results[k][3] <= 1.1e-10
        assert np.array_equal(results[k][0], results[k][1]) and np.array_equal(results[k][0], results[k][2])


def test_threads_launch_one_kernel_with_different_lds():
    """Two threads whose solves take the same kernel, one with 44 KB of LDS per workgroup and one with
    95 KB: each solve gets what it needs whatever the other asked for last."""
    import threading

    systems = [_spd(70001, 8, 50), _spd(400000, 4, 51)]
    results = {0: [], 1: []}

    def work(k):
        c = neon_amd.Context(0)
        try:
            for _ in range(12):
                results[k].append(_solve_csr(c, neon_amd.conjugate_gradient_hip, *systems[k])[0])
        finally:
            c.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in results]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, (A, b) in enumerate(systems):
        assert len(results[k]) == 12
        assert np.linalg.norm(b - A @ results[k][0]) <= 1.1e-10 * np.linalg.norm(b)
        assert all(np.array_equal(x, results[k][0]) for x in results[k])


# a large solve in the launch loop with its one-launch vector part (mixed, FP64) and in the resident grid,
# each a good part of a second long (none reaches its tolerance)
@pytest.mark.parametrize("dims,precision,tol,limit", [((104, 102, 101), "mixed", 1e-30, 6000),
                                                      ((104, 102, 101), "fp64", 1e-30, 3000),
                                                      ((52, 50, 51), "fp64", 1e-150, 8000)])
def test_a_small_solve_takes_turns_with_a_large_one(ctx, dims, precision, tol, limit):
    """Small solves in one thread while a large one, which holds every compute unit, runs in another:
    they get their turn between the large one's batches (2 to 3 ms each; a small solve here takes
    some ten turns) instead of waiting for its end, and neither's result changes."""
    import threading

    print(dims, precision, flush=True)
    large = neon_amd.Context(0)
    try:
        mg, b = _mesh(large, dims, "grid", 0.0)
        if precision == "mixed":
            mg.assemble(neon_amd.PRECISION_MIXED)
            mg.enforce_dirichlet(problems.block_rollers(max(dims), dims=dims).fixed_dofs(), b)
        small, c = _mesh(ctx, (9, 8, 7), "grid", 0.0)
        out = {}

        def solve_large(key):
            try:
                mg.solve(b, tol=tol, max_iterations=limit)
            except neon_amd.computational_error as e:
                out[key] = e.code
            out[key, "u"] = mg.solve(b, tol=1e-6)[0]

        alone = small.solve(c, tol=1e-10)[0]
        solve_large("alone")
        thread = threading.Thread(target=solve_large, args=("shared",))
        thread.start()
        count = 0
        while thread.is_alive():
            assert np.array_equal(small.solve(c, tol=1e-10)[0], alone)
            count += 1
        thread.join()
        print(count, "small solves", flush=True)
        assert out["alone"] == out["shared"] == _capi.NEON_NONCONVERGED
        assert np.array_equal(out["alone", "u"], out["shared", "u"])
        assert count >= 6, count
        del mg
    finally:
        large.close()


def _unsymmetric(n, per_row, seed):
    A, b = _spd(n, per_row, seed)
    rng = np.random.default_rng(seed + 1)
    A = A.copy()
    A.data *= rng.uniform(0.5, 1.0, len(A.data))
    return (A + sp.diags(np.abs(A).sum(axis=1).A1 + 1.0)).tocsr(), b


# BiCGSTAB follows roundoff closely (test_bicgstab_host_csr_parity): counts within 15 % and 3; its
# recurrence residual drifts from the true one by eps |A| |x| per iteration times the largest
# residual on the way, some orders below 1e-10 |b| on these diagonally dominant systems
@pytest.mark.parametrize("n,per_row", [(1, 1), (63, 4), (65, 5), (900, 60), (20000, 30), (262143, 9), (700000, 5)])
def test_bicgstab_on_host_csr(ctx, n, per_row):
    print(n, per_row, flush=True)
    A, b = _unsymmetric(n, per_row, n)
    grid, launches = _both(ctx, lambda: _solve_csr(ctx, neon_amd.biconjugate_gradient_stabilised_hip, A, b))
    for x, its, _ in (grid, launches):
        assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)
    assert abs(grid[1] - launches[1]) <= 3 + 0.15 * launches[1], (grid[1], launches[1])


# the unsymmetric tangent on the full copy with eight and four wavefronts per slice, its share of the
# matrix in registers; several rounds; one wavefront per slice; and a symmetric copy
@pytest.mark.parametrize("dims,model", [((3, 4, 3), "damage"), ((12, 11, 13), "damage"), ((30, 29, 31), "damage"),
                                        ((36, 35, 37), "damage"), ((45, 44, 43), "damage"), ((20, 21, 19), "neohooke")])
def test_bicgstab_on_the_mesh_tangent(ctx, dims, model):
    print(dims, model, flush=True)
    p = problems.block_rollers(max(dims), dims=dims)
    if model == "damage":
        q = problems.damage_cube(1)
        params = np.repeat(q.params[:1], p.n_elem, axis=0)
        mg = neon_amd.DeviceMesh(p.X, p.conn, params, model=neon_amd.MODEL_J2_DAMAGE, context=ctx,
                                 damage=problems.DAMAGE_CONSTANTS)
    else:
        mg = neon_amd.DeviceMesh(p.X, p.conn, p.params, context=ctx)
        mg.update_internal_variables()
    mg.assemble()
    b = np.random.default_rng(12).standard_normal(mg.n_dofs)
    mg.enforce_dirichlet(p.fixed_dofs(), b)
    A = _matrix(mg)
    # the right-hand side of a solution of order one
    b = A @ b
    grid, launches = _both(ctx, lambda: mg.solve(b, solver=neon_amd.SOLVER_BICGSTAB, tol=1e-10))
    for x, its, _ in (grid, launches):
        assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)
    assert abs(grid[1] - launches[1]) <= 3 + 0.15 * launches[1], (grid[1], launches[1])


@pytest.mark.parametrize("criterion", [neon_amd.STOP_RELATIVE, neon_amd.STOP_ABSOLUTE_PRECONDITIONED])
def test_bicgstab_ends(ctx, criterion):
    """The CUDA rule's early exit (an identity matrix), a zero right-hand side, the iteration limit
    inside and past a launch, and values that are not finite end as they do by launches."""
    cls = neon_amd.biconjugate_gradient_stabilised_hip

    def outcome(A, b, tol, limit):
        got = []
        for timed in (False, True):
            s = cls(tol, limit, criterion=criterion, context=ctx)
            x = np.zeros(len(b))
            ctx.profile(timed)
            try:
                s.solve(A, x, b)
                code = 0
            except neon_amd.computational_error as e:
                code = e.code
            finally:
                ctx.profile(False)
            got.append((code, s.iterations))
        assert got[0] == got[1], got
        return got[0]

    ident = sp.identity(500, format="csr")
    b = np.linspace(1.0, 2.0, 500)
    assert outcome(ident, b, 1e-10, 100)[0] in (0, _capi.NEON_BREAKDOWN, _capi.NEON_NAN_OR_INF)
    assert outcome(ident, np.zeros(500), 1e-10, 100) == (0, 0)
    A, b = _unsymmetric(2000, 12, 4)
    assert outcome(A, b, 1e-30, 3) == (_capi.NEON_NONCONVERGED, 3)
    b[5] = np.nan
    assert outcome(A, b, 1e-10, 100)[0] == _capi.NEON_NAN_OR_INF
