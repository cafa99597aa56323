"""Batched stepping (several simulations, each solve kind in one persistent
launch for all of them) against stepping the same simulations one by one,
and the autotuner of the batched solves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(gpu, specs, precision, rtol):
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation

    sims = []
    for n, lid, nu in specs:
        sims.append(Simulation(mesh.cavity(n, lid_speed=lid), nu, 0.005, device=gpu, rtol=rtol,
                               precision=precision))
    return sims


SPECS = [(8, 1.0, 0.01), (20, 0.7, 0.002), (12, 1.9, 0.005), (16, 1.2, 0.001), (10, 0.5, 0.008)]


@pytest.mark.parametrize("resident", ["1", "0"])
@pytest.mark.parametrize("precision", ["fp64", "fp32_refined"])
def test_batch_matches_individual_steps(gpu, monkeypatch, capfd, precision, resident):
    from navier_stokes_fem_amd.simulation import step_batch

    monkeypatch.setenv("NSFEM_CG_RESIDENT", resident)
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    # the FP32 form is run at 1e-9: on these tiny systems a tighter
    # tolerance exhausts the default iteration limit (the row count)
    rtol = 1e-11 if precision == "fp64" else 1e-9
    tol = 1e-8 if precision == "fp64" else 1e-6
    one = _batch(gpu, SPECS, precision, rtol)
    many = _batch(gpu, SPECS, precision, rtol)
    for s in one:
        s.step(4)
    capfd.readouterr()
    stats = step_batch(many, 4)
    form = {cols: waves > 0 for _, cols, waves in _launches(capfd.readouterr().err)}
    assert form == {1: resident == "1", 2: resident == "1" and precision == "fp64"}
    assert len(stats) == len(SPECS)
    for a, b, st in zip(one, many, stats):
        assert st["steps"] == 4
        assert max(st["max_relative_residual"]) <= rtol * 1.01
        for fa, fb in zip(a.fields(), b.fields()):
            np.testing.assert_allclose(fb, fa, rtol=0, atol=tol * max(1.0, np.abs(fa).max()))
    for s in one + many:
        s.close()


def test_batch_autotune_keeps_results(gpu):
    from navier_stokes_fem_amd.simulation import autotune_batch, step_batch

    ref = _batch(gpu, SPECS, "fp64", 1e-11)
    tuned = _batch(gpu, SPECS, "fp64", 1e-11)
    t = autotune_batch(tuned)
    print("autotune:", t)
    assert t["rows_per_wave"] in (64, 32, 16) and t["block_scale"] in (1, 2, 4)
    assert t["velocity_block_scale"] in (1, 2, 4)
    assert t["seconds_per_iteration"] > 0
    step_batch(ref, 3)
    step_batch(tuned, 3)
    for a, b in zip(ref, tuned):
        for fa, fb in zip(a.fields(), b.fields()):
            np.testing.assert_allclose(fb, fa, rtol=0, atol=1e-8 * max(1.0, np.abs(fa).max()))
    for s in ref + tuned:
        s.close()


def test_batch_of_many_small_instances(gpu):
    """More instances than a block each would need: 40 cavities of 4..12."""
    from navier_stokes_fem_amd.simulation import step_batch

    rng = np.random.default_rng(5)
    specs = [(int(rng.integers(4, 13)), float(rng.uniform(0.5, 2)), 0.01) for _ in range(40)]
    sims = _batch(gpu, specs, "fp64", 1e-10)
    stats = step_batch(sims, 2)
    for st in stats:
        assert max(st["max_relative_residual"]) <= 1e-10 * 1.01
    # one of them stepped alone gives the same fields
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation

    n, lid, nu = specs[7]
    alone = Simulation(mesh.cavity(n, lid_speed=lid), nu, 0.005, device=gpu, rtol=1e-10)
    alone.step(2)
    for fa, fb in zip(alone.fields(), sims[7].fields()):
        np.testing.assert_allclose(fb, fa, rtol=0, atol=1e-7 * max(1.0, np.abs(fa).max()))
    alone.close()
    for s in sims:
        s.close()


@pytest.mark.parametrize("levels", [False, True])
def test_batch_coarse_correction(gpu, levels):
    """Coarse corrections of several instances share one batched launch:
    every solve meets the tolerance, the instance without a coarse space (odd
    n) runs no coarse solve, the pressure solves of the others take fewer
    iterations than the same batch without coarse spaces (six steps from
    rest on small meshes: a few per cent), and the fields
    match the same simulations with the same coarse spaces stepped one by one
    (FP64 at 1e-11, to 1e-7 of the field scale).  With `levels` the 64^2
    and 96^2 instances also get a multigrid level below their coarse space
    and solve their coarse systems by V-cycles, while the 48^2 one stays in
    the batched coarse CG."""
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import step_batch

    specs = [(64, 1.0, 1e-3), (48, 0.7, 2e-3), (33, 1.5, 1e-3), (96, 1.2, 1e-3)]
    rtol = 1e-11

    def with_coarse(sims):
        for (n, _, _), s in zip(specs, sims):
            if n % 2 == 0:
                s.set_coarse_space(mesh.cavity_prolongation(n, 2))
                if levels and n != 48:
                    s.add_coarse_level(mesh.cavity_prolongation(n // 2, 2))
        return sims

    plain = _batch(gpu, specs, "fp64", rtol)
    batched = with_coarse(_batch(gpu, specs, "fp64", rtol))
    one = with_coarse(_batch(gpu, specs, "fp64", rtol))
    st_p = step_batch(plain, 6)
    st_c = step_batch(batched, 6)
    for s in one:
        s.step(6)
    its_p = sum(st["cg_iterations"][2] for (n, _, _), st in zip(specs, st_p) if n % 2 == 0)
    its_c = sum(st["cg_iterations"][2] for (n, _, _), st in zip(specs, st_c) if n % 2 == 0)
    print(f"pressure iterations of the instances with a coarse space: {its_p} -> {its_c}; "
          f"coarse {[st['coarse_iterations'] for st in st_c]}")
    for (n, _, _), st in zip(specs, st_c):
        assert max(st["max_relative_residual"]) <= rtol * 1.01
        assert (st["coarse_iterations"] > 0) == (n % 2 == 0)
    assert its_c < its_p  # a few % this early; the single-mesh tests measure the gain
    for a, b in zip(one, batched):
        for fa, fb in zip(a.fields(), b.fields()):
            np.testing.assert_allclose(fb, fa, rtol=0, atol=1e-7 * max(1.0, np.abs(fa).max()))
    for s in plain + batched + one:
        s.close()


def _launches(err):
    """(instances, columns, waves of a resident block or 0) of each batched CG
    launch, in order."""
    out = []
    for line in err.splitlines():
        if "cg batch launch" in line:
            f = dict(w.split("=") for w in line.split() if "=" in w)
            out.append((int(f["instances"]), int(f["cols"]),
                        int(f["waves"]) if f["resident"] != "0" else 0))
    return out


# pressure systems of one wave tile, of one block with one, two, three and
# four tiles a wave, and of several blocks of two and three
REFINED = [(4, 1.0, 0.01), (20, 0.7, 0.002), (40, 1.1, 0.003), (47, 1.2, 0.001), (55, 1.9, 0.005),
           (90, 0.5, 0.008), (128, 1.4, 0.002)]


def _steps(gpu, specs, precision, steps, capfd):
    from navier_stokes_fem_amd.simulation import step_batch

    sims = _batch(gpu, specs, precision, 1e-8)
    capfd.readouterr()
    stats = step_batch(sims, steps)
    launches = _launches(capfd.readouterr().err)
    fields = [s.fields() for s in sims]
    for s in sims:
        s.close()
    return fields, [(st["cg_iterations"], st["cg_refinements"]) for st in stats], launches


@pytest.mark.parametrize("specs", [REFINED[:1], REFINED[:3], REFINED[:4], REFINED],
                         ids=["1", "3", "4", "7"])
def test_refined_batch_equals_streaming(gpu, monkeypatch, capfd, specs):
    """A refined batch's pressure solves run resident on the blocks and waves
    of the streaming form, its two-column solves stream: the same sums either
    way, so fields and counts are those of the streaming batch bit for bit."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    got, its, launches = _steps(gpu, specs, "fp32_refined", 2, capfd)
    assert launches == 2 * [(len(specs), 2, 0), (len(specs), 1, 16), (len(specs), 2, 0)]
    monkeypatch.setenv("NSFEM_CG_RESIDENT", "0")
    want, ref, launches = _steps(gpu, specs, "fp32_refined", 2, capfd)
    assert not any(waves for _, _, waves in launches)
    assert its == ref
    for a, b in zip(got, want):
        for fa, fb in zip(a, b):
            np.testing.assert_array_equal(fa, fb)


def test_refined_batch_past_the_device(gpu, monkeypatch, capfd):
    """Far more blocks wanted than the device has: the 100^2 systems' one block
    each would have ten tiles a wave, so the pressure solves take the resident
    form's own split, in two launches (12 systems of at least 22 blocks): every solve meets its
    tolerance, and the fields are the streaming batch's to what solves to 1e-8
    leave (measured 1e-3 of the fields' norm against a tight solve; either
    side's is half of the bar)."""
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    specs = [(n, 1.0, 0.004) for n in 12 * (256,) + (100, 100, 96, 20)]
    got, _, launches = _steps(gpu, specs, "fp32_refined", 1, capfd)
    pressure = [(i, waves) for i, cols, waves in launches if cols == 1]
    assert len(pressure) == 2 and sum(i for i, _ in pressure) == len(specs)
    assert {w for _, w in pressure} == {12}
    monkeypatch.setenv("NSFEM_CG_RESIDENT", "0")
    want, _, launches = _steps(gpu, specs, "fp32_refined", 1, capfd)
    assert not any(waves for _, _, waves in launches)
    for a, b in zip(got, want):
        for fa, fb in zip(a, b):
            assert np.linalg.norm(fa - fb) <= 2e-3 * np.linalg.norm(fb)


def _shuffled(n, seed):
    """The n^2 cavity with its pressure nodes in random order: no window of
    rows holds the columns of a block's."""
    from navier_stokes_fem_amd import mesh

    m = mesh.cavity(n)
    old = np.arange(m.node_count)
    old[:m.pressure_count] = np.random.default_rng(seed).permutation(m.pressure_count)
    new = np.empty_like(old)
    new[old] = np.arange(m.node_count)
    return mesh.Mesh(nodes=m.nodes[old], elements=new[m.elements].astype(m.elements.dtype),
                     pressure_count=m.pressure_count,
                     vel_bc_nodes=new[m.vel_bc_nodes].astype(m.vel_bc_nodes.dtype),
                     vel_bc_u=m.vel_bc_u, vel_bc_v=m.vel_bc_v,
                     p_bc_nodes=new[m.p_bc_nodes].astype(m.p_bc_nodes.dtype),
                     p_bc_values=m.p_bc_values, name=m.name, info=m.info, grid=None)


@pytest.mark.parametrize("precision", ["fp64", "fp32_refined"])
def test_batch_with_a_system_that_streams(gpu, monkeypatch, capfd, precision):
    """A pressure system past the resident form's window sends its launch to
    the streaming form; every solve meets its tolerance and the instances match
    the same simulations stepped alone (solves to 1e-9, as in
    test_batch_matches_individual_steps)."""
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation, step_batch

    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    n = 126 if precision == "fp64" else 180  # 8 and 4 bytes a row of the window
    meshes = [mesh.cavity(12), _shuffled(n, 1), mesh.cavity(20)]
    one, many = ([Simulation(m, 0.01, 0.005, device=gpu, rtol=1e-9, precision=precision)
                  for m in meshes] for _ in range(2))
    for s in one:
        s.step(1)
    capfd.readouterr()
    stats = step_batch(many, 1)
    launches = _launches(capfd.readouterr().err)
    assert (3, 1, 0) in launches and (3, 1, 12) not in launches and (3, 1, 16) not in launches
    for a, b, st in zip(one, many, stats):
        assert max(st["max_relative_residual"]) <= 1e-9 * 1.01
        for fa, fb in zip(a.fields(), b.fields()):
            assert np.linalg.norm(fa - fb) <= 1e-3 * np.linalg.norm(fa)
    for s in one + many:
        s.close()


@pytest.mark.parametrize("resident", ["1", "0"])
def test_batch_of_more_instances_than_blocks(gpu, monkeypatch, capfd, resident):
    """270 instances: a second launch in either form, with the same fields as
    alone."""
    from navier_stokes_fem_amd import mesh
    from navier_stokes_fem_amd.simulation import Simulation, step_batch

    monkeypatch.setenv("NSFEM_CG_RESIDENT", resident)
    monkeypatch.setenv("NSFEM_CG_VERBOSE", "1")
    specs = [(2 + k % 4, 1.0 + k / 270.0, 0.01) for k in range(270)]
    sims = _batch(gpu, specs, "fp64", 1e-10)
    capfd.readouterr()
    stats = step_batch(sims, 1)
    launches = _launches(capfd.readouterr().err)
    assert all((waves > 0) == (resident == "1") for _, _, waves in launches)
    assert len(launches) == 6 and sum(i for i, _, _ in launches) == 3 * 270
    for k in (0, 3, 255, 256, 269):
        assert max(stats[k]["max_relative_residual"]) <= 1e-10 * 1.01
        n, lid, nu = specs[k]
        alone = Simulation(mesh.cavity(n, lid_speed=lid), nu, 0.005, device=gpu, rtol=1e-10)
        alone.step(1)
        for fa, fb in zip(alone.fields(), sims[k].fields()):
            np.testing.assert_allclose(fb, fa, rtol=0, atol=1e-7 * max(1.0, np.abs(fa).max()))
        alone.close()
    for s in sims:
        s.close()
