"""The resident form of the CG (the matrix in the blocks' registers, p in an
LDS window, the sums and q crossing blocks at the coherence point) against the
streaming forms, at the sizes where its tiles, windows and grids end.

The one-column mixed form has the streaming form's products, sums and grid:
bit-identical.  The others reach the same tolerance by another order of sums:
the true residual is checked, and the iteration counts agree to a few."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banded(n, offsets, seed, empty=()):
    """A strictly diagonally dominant symmetric matrix with these sub- and
    superdiagonals; rows in `empty` hold their diagonal alone."""
    rng = np.random.default_rng(seed)
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [np.full(n, 1.0 + 2.02 * len(offsets))]
    lone = np.zeros(n, bool)
    lone[[e for e in empty if e < n]] = True
    for o in offsets:
        i = np.arange(max(n - o, 0))
        i = i[~lone[i] & ~lone[i + o]]
        v = -rng.uniform(0.5, 1.0, len(i))
        rows += [i, i + o]
        cols += [i + o, i]
        vals += [v, v]
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    order = np.lexsort((c, r))
    rs = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(r, minlength=n), out=rs[1:])
    return rs.astype(np.int32), c[order].astype(np.int32), v[order]


def solve(gpu, A, b, x0, columns, precision, capfd, rtol=1e-10, max_iterations=-1):
    gpu.upload_csr(6, *A)
    bb, bx = gpu.buffer(b), gpu.buffer(x0)
    capfd.readouterr()
    st = gpu.cg_solve(6, bb, bx, columns=columns, rtol=rtol, precision=precision,
                      max_iterations=max_iterations, raise_on_error=False)
    resident = "resident=0" not in capfd.readouterr().err
    x = bx.download()
    bb.close()
    bx.close()
    return x, st, resident


# (rows, off-diagonals): one row; less than a wave; the edges of a wave tile;
# two and three tiles a wave of one block; several blocks with windows that
# reach past them; rows of 19 nonzeros (the long-row kernels), 20 and of all
# lengths
SYSTEMS = [(1, ()), (2, (1,)), (63, (1, 5)), (64, (1, 5)), (65, (1, 5)), (767, (1, 2, 30)),
           (1600, (1, 40, 41)), (6000, (1, 60, 61)), (20011, (1, 140, 141)),
           (1100, tuple(range(1, 10))), (9000, (1, 2, 3, 90, 91, 92, 180, 181, 182)),
           (700, (1, 2, 3, 4, 5, 6, 7, 8, 600))]


@pytest.mark.parametrize("columns,precision", [(1, "fp64"), (2, "fp64"), (1, "fp32_refined"),
                                               (2, "fp32_refined")])
@pytest.mark.parametrize("n,offsets", SYSTEMS, ids=lambda v: str(v) if isinstance(v, int) else None)
def test_resident_equals_streaming(gpu, oracle, monkeypatch, capfd, n, offsets, columns, precision):
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    A = banded(n, offsets, n, empty=(0, 64, 65, 1023))
    rng = np.random.default_rng(n + 1)
    b = rng.standard_normal(columns * n)
    b[n:] *= 7.0
    x0 = 0.1 * rng.standard_normal(columns * n)
    got, st, resident = solve(gpu, A, b, x0, columns, precision, capfd, max_iterations=1000)
    assert resident
    monkeypatch.setenv("NSFEM_CG_RESIDENT", "0")
    want, ref, resident = solve(gpu, A, b, x0, columns, precision, capfd, max_iterations=1000)
    assert not resident
    if columns == 1 and precision == "fp32_refined":
        np.testing.assert_array_equal(got, want)
        assert [s["iterations"] for s in st] == [s["iterations"] for s in ref]
        assert [s["refinements"] for s in st] == [s["refinements"] for s in ref]
    for c in range(columns):
        bc, xc = b[c * n:(c + 1) * n], got[c * n:(c + 1) * n]
        assert st[c]["status"] == 0 and ref[c]["status"] == 0
        r = np.linalg.norm(oracle.spmv_sub(A, bc, xc))
        assert r <= 1e-10 * np.linalg.norm(bc) * (1 + 1e-9)
        assert abs(st[c]["final_residual"] - r) <= 1e-3 * r + 1e-13 * np.linalg.norm(bc)
        assert abs(st[c]["iterations"] - ref[c]["iterations"]) <= 2 + 0.1 * ref[c]["iterations"]
        assert st[c]["rhs_norm"] == pytest.approx(ref[c]["rhs_norm"], rel=1e-13)
        assert st[c]["initial_residual"] == pytest.approx(ref[c]["initial_residual"], rel=1e-12)


@pytest.mark.parametrize("grid", ["1", "3", "97", "256"])
def test_resident_grids(gpu, oracle, monkeypatch, capfd, grid):
    """One system over few and many blocks, at most one wave tile a wave and
    several words a polling lane."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    n = 3000 if grid == "1" else 8500 if grid == "3" else 30011
    A = banded(n, (1, 170, 171), 5)
    b = np.random.default_rng(6).standard_normal(n)
    monkeypatch.setenv("NSFEM_CG_GRID", grid)
    for precision in ("fp64", "fp32_refined"):
        x, st, resident = solve(gpu, A, b, np.zeros(n), 1, precision, capfd)
        assert resident and st[0]["status"] == 0
        assert np.linalg.norm(oracle.spmv_sub(A, b, x)) <= 1e-10 * np.linalg.norm(b) * (1 + 1e-9)


def test_systems_that_stay_streaming(gpu, monkeypatch, capfd):
    """A row of 21 nonzeros, a window past the LDS and an explicit streaming
    form keep the streaming kernels."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    b = np.random.default_rng(7).standard_normal(60000)
    for n, offsets in ((500, tuple(range(1, 11))), (60000, (1, 30000))):
        A = banded(n, offsets, 8)
        _, st, resident = solve(gpu, A, b[:n], np.zeros(n), 1, "fp64", capfd)
        assert not resident and st[0]["status"] == 0
    A = banded(500, (1, 9), 9)
    monkeypatch.setenv("NSFEM_CG_PHASE", "items")
    _, st, resident = solve(gpu, A, b[:500], np.zeros(500), 1, "fp32_refined", capfd)
    assert not resident and st[0]["status"] == 0


@pytest.mark.parametrize("columns,precision", [(1, "fp64"), (2, "fp64"), (1, "fp32_refined"),
                                               (2, "fp32_refined")])
def test_resident_ends_as_streaming(gpu, monkeypatch, capfd, columns, precision):
    """Ends other than convergence: the iteration limit with the last iterate,
    a matrix that is not positive definite, a zero right-hand side, a guess
    that is the solution, infinities and NaN in the right-hand side."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    n = 4000
    A = banded(n, (1, 50, 51), 11)
    neg = (A[0], A[1], -A[2])
    rng = np.random.default_rng(12)
    b = rng.standard_normal(columns * n)
    zero = np.zeros(columns * n)
    inf, nan = b.copy(), b.copy()
    inf[17] = np.inf
    nan[-5] = np.nan
    cases = [(A, b, zero, 3), (neg, b, zero, -1), (A, zero, zero, -1), (A, zero, b, -1),
             (A, inf, zero, 40), (A, nan, zero, 40)]
    for i, (M, rhs, x0, limit) in enumerate(cases):
        monkeypatch.delenv("NSFEM_CG_RESIDENT", raising=False)
        got, st, resident = solve(gpu, M, rhs, x0, columns, precision, capfd, 1e-12, limit)
        assert resident
        monkeypatch.setenv("NSFEM_CG_RESIDENT", "0")
        want, ref, _ = solve(gpu, M, rhs, x0, columns, precision, capfd, 1e-12, limit)
        assert [s["status"] for s in st] == [s["status"] for s in ref], i
        assert [s["iterations"] for s in st] == [s["iterations"] for s in ref], i
        same = np.isfinite(got) == np.isfinite(want)
        assert same.all(), i
        fine = np.isfinite(want)
        # a few steps from the same start: only the sums' order differs
        np.testing.assert_allclose(got[fine], want[fine], rtol=1e-4 if i == 1 else 1e-6,
                                   atol=1e-9 * (1 + np.abs(want[fine]).max(initial=0.0)))


@pytest.mark.parametrize("n,rule", [(20000, "one"), (36000, "two"), (60000, "two"), (100000, "one")])
def test_streaming_blocks_of_long_rows(gpu, oracle, monkeypatch, capfd, n, rule):
    """One-column refined solves past the resident window: one wave tile a
    wave up to 96 blocks and where two tiles need more than 128, else two
    (tiles of some 28 rows of 19 nonzeros)."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    A = banded(n, (1, 2, 3, 4, 5, 6, 7, 8, n // 2), 31)
    b = np.random.default_rng(32).standard_normal(n)
    gpu.upload_csr(6, *A)
    x = gpu.buffer(np.zeros(n))
    capfd.readouterr()
    st = gpu.cg_solve(6, gpu.buffer(b), x, rtol=1e-10, precision="fp32_refined")[0]
    line = [v for v in capfd.readouterr().err.splitlines() if "cg launch" in v][0]
    f = dict(w.split("=") for w in line.split() if "=" in w)
    tiles = int(line.split("wave tiles=")[1].split()[0])
    one, two = tiles // 12, tiles // 24
    assert rule == ("one" if one <= 96 or two > 128 else "two")
    assert f["resident"] == "0"
    assert int(f["grid"]) == min(int(f["maxgrid"]), one if rule == "one" else two)
    assert st["status"] == 0
    assert np.linalg.norm(oracle.spmv_sub(A, b, x.download())) <= 1e-10 * np.linalg.norm(b) * (1 + 1e-9)


def test_windows_of_two_handles(gpu, monkeypatch, capfd):
    """Two device handles solve by turns with the same kernel, one with a
    window of some 100 KB of LDS, the other of some 50: what a kernel may take
    is not one solve's."""
    from navier_stokes_fem_amd.device import GPUSimulationDevice

    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    other = GPUSimulationDevice(0)
    systems = [(gpu, banded(12000, (1, 2500), 21)), (other, banded(12000, (1, 1200), 22))]
    b = np.random.default_rng(23).standard_normal(12000)
    first = [None, None]
    for turn in range(3):
        for k, (dev, A) in enumerate(systems):
            x, st, resident = solve(dev, A, b, np.zeros(12000), 1, "fp64", capfd)
            assert resident and st[0]["status"] == 0
            if turn == 0:
                first[k] = x
            np.testing.assert_array_equal(x, first[k])


# (scale of the matrix, scale of the solution): (q, q) underflows; alpha^2
# overflows; (q, q) overflows while (r, r) and (p, q) do not; the residual's
# own squares leave the range
SCALES = [(1e-170, 1.0), (1e-170, 1e100), (1e150, 1e-75), (1e150, 1e-160), (1e-60, 1e-100),
          (1e160, 1e-80), (2.0 ** 300, 2.0 ** -200)]


@pytest.mark.parametrize("columns", [1, 2])
@pytest.mark.parametrize("n", [700, 9000])
@pytest.mark.parametrize("matrix,solution", SCALES)
def test_scales_past_the_recurrence(gpu, oracle, monkeypatch, capfd, n, columns, matrix, solution):
    """FP64 at scales where the next (r, r) cannot be formed from (r, q) and
    (q, q): the solve ends as the streaming one, which adds (r, r) itself."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    A = banded(n, (1, 30, 31), n)
    A = (A[0], A[1], A[2] * matrix)
    x = np.random.default_rng(n).standard_normal(columns * n) * solution
    zero = np.zeros(n)
    b = np.concatenate([oracle.spmv_sub(A, zero, -x[c * n:(c + 1) * n]) for c in range(columns)])
    got, st, _ = solve(gpu, A, b, np.zeros(columns * n), columns, "fp64", capfd)
    monkeypatch.setenv("NSFEM_CG_RESIDENT", "0")
    want, ref, _ = solve(gpu, A, b, np.zeros(columns * n), columns, "fp64", capfd)
    assert [s["status"] for s in st] == [s["status"] for s in ref]
    assert [s["iterations"] for s in st] == pytest.approx([s["iterations"] for s in ref], abs=2)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-8 * solution)


def test_scales_past_the_recurrence_in_a_batch(gpu, monkeypatch, capfd):
    """Two of a batch's systems leave the recurrence's range ((q, q) below
    1e-290): they run alone in the streaming form, the third stays."""
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation, step_batch

    out = []
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    for resident in ("1", "0"):
        monkeypatch.setenv("NSFEM_CG_RESIDENT", resident)
        sims = [Simulation(mesh.cavity(n, lid_speed=lid), 1e-3, 5e-3, device=gpu, rtol=1e-6,
                           precision="fp64") for n, lid in ((12, 1e-144), (16, 1.0), (20, 1e-144))]
        capfd.readouterr()
        stats = step_batch(sims, 2)
        alone = [line for line in capfd.readouterr().err.splitlines() if "cg launch" in line]
        assert bool(alone) == (resident == "1")
        assert all("resident=0" in line for line in alone)
        out.append(([s.fields() for s in sims], [st["cg_iterations"] for st in stats]))
        for s in sims:
            s.close()
    (got, its), (want, ref) = out
    for a, b, i, j in zip(got, want, its, ref):
        assert np.abs(np.subtract(i, j)).max() <= 4
        for fa, fb in zip(a, b):
            np.testing.assert_allclose(fa, fb, rtol=0, atol=1e-3 * np.abs(fb).max())
