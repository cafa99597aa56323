"""The V-cycle preconditioned chain at the sizes where its kernels' blocks and
loops end: whole steps against the oracle's, every solve to 1e-10, with the
smoke test's bar (1e-6 of the fields' scale; the solves leave about
cond * 1e-10, the point location is the same)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _chain(gpu, m, precision, min_size):
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation

    s = Simulation(m, 0.01, 0.01, device=gpu, rtol=1e-10, precision=precision,
                   velocity_jacobi="mass")
    levels = mesh.grid_hierarchy(m, min_size=min_size)
    s.set_coarse_space(levels[0], rtol=1e-6)
    for level in levels[1:]:
        s.add_coarse_level(level)
    s.set_pressure_multigrid(True)
    s.set_velocity_multigrid(mesh.velocity_hierarchy(m, min_size=min_size), mode=2)
    s.set_velocity_projection(2)
    s.set_mass_projection(1)
    return s


# deepest pressure / velocity levels of the cavity: 8 and 1 nodes (less than a
# wave), 323 and 256 (the dense product's last loop alone), 675 and 576 (one
# whole round of its unrolled loop and a rest), 1,088 and 961 (two and one);
# 66: 1,155 pressure nodes, solved by CG in place of a dense inverse
@pytest.mark.parametrize("precision", ["fp64", "fp32_refined"])
@pytest.mark.parametrize("n,min_size", [(4, 2), (34, 17), (50, 17), (64, 17), (66, 17)])
def test_chain_step_against_oracle(gpu, oracle, n, min_size, precision):
    from navier_stokes_fem_amd import mesh

    m = mesh.cavity(n)
    s = _chain(gpu, m, precision, min_size)
    st = s.step(2)
    got = s.fields()
    s.close()
    asm = oracle.Assembly(m, 0.01, 0.01)
    tree = oracle.kd_build(m.xy(), m.elems())
    want = oracle.initial_fields(m)
    for _ in range(2):
        want = oracle.step(asm, tree, m, 0.01, *want, rtol=1e-10)[:3]
    scale = max(np.abs(f).max() for f in want)
    for a, b in zip(got, want):
        assert np.abs(a - b).max() < 1e-6 * scale
    assert st["vcycle_solves"][:3] == [2, 2, 2]
    assert max(st["vcycle_iterations"][:3]) <= 2 * 20


# a basis of one vector (the plain dot), of the most that one launch of dots
# takes (8), one more, and two launches and one more; 961 velocity nodes end
# inside the first block's chunk of 1,024, 1,089 in the second's
@pytest.mark.parametrize("depth", [1, 8, 9, 17])
@pytest.mark.parametrize("n", [15, 16])
def test_projection_basis_at_its_edges(gpu, n, depth):
    """The projection changes only where a solve starts: past a restart of
    the basis the fields are those of the run without it to what solves to
    1e-11 leave (cond * 1e-11 of a cavity this small is far below 1e-6), and
    the diffusion solves take fewer iterations (a basis whose coefficients
    were wrong in any vector would start them further away)."""
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation

    m = mesh.cavity(n)
    out = []
    for d in (0, depth):
        s = Simulation(m, 1e-3, 1e-3, device=gpu, rtol=1e-11, precision="fp64")
        s.set_velocity_projection(d)
        s.set_mass_projection(d)
        st = s.step(depth + 4)
        out.append((st, s.fields()))
        s.close()
    (s0, f0), (s1, f1) = out
    assert max(s1["max_relative_residual"]) <= 1e-11 * (1 + 1e-6)
    scale = max(np.abs(f).max() for f in f0)
    for a, b in zip(f1, f0):
        assert np.abs(a - b).max() < 1e-6 * scale
    d0, d1 = (sum(s["cg_iterations"][:2]) for s in (s0, s1))
    print(f"diffusion iterations {d0} -> {d1}")
    assert d1 < d0
