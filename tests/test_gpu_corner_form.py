"""The corner form (box cells, blocks of 5 to 8 species: a lane per cell and
corner, coefficients evaluated at the linearisation point inside the apply)
against the oracle: residual, Jacobian apply, diagonal blocks (through steps
with both Jacobi forms), batches; at sides around the tiles' 7, 31 and 63
vertices, odd sizes, non-square boxes and spacings, a compartment that covers
a part of the grid, interface terms, cross-diffusion, diffusion per axis, and
reactions that read time and position.  Sums run in another order than the
oracle's in FP64: 1e-12 relative for one application, the parity bar of 1e-8
for converged steps."""
import numpy as np
import pytest

from tests.oracle_lib import OracleModel, rel_l2_per_species

pytestmark = pytest.mark.gpu

PTS = ("model.time_step_operator.linear_solver.storage = points\n"
       "model.time_step_operator.linear_solver.preconditioner.type = Jacobi\n")


def _ini(dim, cells, species, compartments="domain.expression = 1", extensions=(1.0, 1.0, 1.0), rk="ImplicitEuler",
         extra=""):
    """A chain s0 -> s1 -> ... with one binary reaction per neighbour pair, cross-diffusion of s0 by s1, diffusion per
    axis for s1, and reactions that read time and position."""
    out = [f"[grid]\ndimension = {dim}\ncells = {' '.join(map(str, cells[:dim]))}\n"
           f"extensions = {' '.join(map(str, extensions[:dim]))}\ncell_type = cube",
           "[parser_context]\nkf.type = constant\nkf.value = 0.7", f"[compartments]\n{compartments}"]
    for i in range(species):
        a, b = f"s{i}", f"s{(i + 1) % species}"
        out += [f"[model.scalar_field.{a}]", "compartment = domain", f"storage.expression = {1.0 + 0.1 * i}",
                f"initial.expression = 0.5 + 0.1*sin({i + 1}*position_x + 2*position_y)",
                f"reaction.expression = kf*{b}*{b} - {a}*{b} + 0.1*position_x*{a} + 0.05*time*{b}",
                f"reaction.jacobian.{a}.expression = -{b} + 0.1*position_x",
                f"reaction.jacobian.{b}.expression = 2*kf*{b} - {a} + 0.05*time"]
        if i == 1:
            out.append(f"cross_diffusion.{a}.type = tensor")
            out += [f"cross_diffusion.{a}.{k}{k}.expression = {0.002 * (n + 1)}" for n, k in enumerate("xyz"[:dim])]
        else:
            out.append(f"cross_diffusion.{a}.expression = {0.001 * (i + 1)}")
        if i == 0:
            out.append("cross_diffusion.s1.expression = 0.0004")
    ini = "\n".join(out) + "\n" + extra
    return ini + (f"\n[model.time_step_operator]\ntype = {rk}\nlinear_solver.type = BiCGSTAB\n"
                  "linear_solver.convergence_condition.relative_tolerance = 1e-12\n"
                  "linear_solver.convergence_condition.iteration_range = 1 2000\n"
                  "linear_solver.preconditioner.type = Jacobi\n"
                  "nonlinear_solver.convergence_condition.relative_tolerance = 1e-20\n"
                  "nonlinear_solver.convergence_condition.absolute_tolerance = 1e-28\n"
                  "nonlinear_solver.convergence_condition.iteration_range = 0 40\n")


SHAPES = [(2, (1, 1)), (2, (5, 3)), (2, (30, 31)), (2, (63, 14)), (2, (70, 33)), (3, (1, 1, 1)), (3, (3, 6, 7)),
          (3, (7, 8, 6)), (3, (15, 4, 9))]


@pytest.mark.parametrize("species", [5, 6, 8])
@pytest.mark.parametrize("dim,cells", SHAPES)
def test_residual_and_apply(dca, dim, cells, species):
    print(f"case: corner form {dim}D {cells} {species} species", flush=True)
    ini = _ini(dim, cells, species, extensions=(1.0, 0.6, 1.7))
    orc = OracleModel(ini)
    rng = np.random.default_rng(species)
    x = v = None
    for tile in ("0", "1"):
        gpu = dca.Model(ini, PTS + f"model.time_step_operator.linear_solver.point_tile = {tile}\n", 0)
        if x is None:
            x, v = 0.5 + 0.2 * rng.random(gpu.n_dof), rng.standard_normal(gpu.n_dof)
        for cm, ca in ((1.0, 0.0), (0.0, 0.7), (1.0, 0.3)):
            ro, vals = orc.assemble(x, 0.4, cm, ca)
            r, _ = gpu.assemble(x, 0.4, cm, ca, jacobian=False)
            assert np.abs(r - ro).max() <= 1e-12 * np.abs(ro).max()
            ref = orc.csr(vals) @ v
            y = gpu.jacobian_apply(x, 0.4, cm, ca, v)
            assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
        gpu.close()
    orc.close()


@pytest.mark.parametrize("dim,cells,species", [(d, c, b) for d, c in SHAPES for b in (5, 6)] +
                         [(2, (30, 31), 8), (2, (70, 33), 8), (3, (15, 4, 9), 8)])
def test_default_storage(dca, dim, cells, species):
    """The same on the storage that a model takes by itself, which is the evaluated form at these sizes."""
    print(f"case: corner form by default {dim}D {cells} {species} species", flush=True)
    ini = _ini(dim, cells, species, extensions=(1.0, 0.6, 1.7))
    orc = OracleModel(ini)
    rng = np.random.default_rng(species)
    x = v = None
    for tile in ("0", "1"):
        gpu = dca.Model(ini, f"model.time_step_operator.linear_solver.point_tile = {tile}\n", 0)
        assert "dcg_tile_0_e0" in gpu.generated_source()
        if x is None:
            x, v = 0.5 + 0.2 * rng.random(gpu.n_dof), rng.standard_normal(gpu.n_dof)
        for cm, ca in ((1.0, 0.0), (0.0, 0.7), (1.0, 0.3)):
            ro, vals = orc.assemble(x, 0.4, cm, ca)
            r, _ = gpu.assemble(x, 0.4, cm, ca, jacobian=False)
            assert np.abs(r - ro).max() <= 1e-12 * np.abs(ro).max()
            ref = orc.csr(vals) @ v
            y = gpu.jacobian_apply(x, 0.4, cm, ca, v)
            assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
        gpu.close()
    orc.close()


@pytest.mark.parametrize("runtime", [False, True])
@pytest.mark.parametrize("precond", ["Jacobi", "VertexBlockJacobi"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim,cells", [(2, (33, 20)), (3, (9, 8, 6))])
def test_steps(dca, dim, cells, precision, precond, runtime):
    """A ball compartment (its rows have partial stencils, its vertices are not the grid's), two stages."""
    print(f"case: corner form steps {dim}D {precision} {precond} runtime={runtime}", flush=True)
    r2 = " + ".join(f"(position_{a}-0.5)^2" for a in "xyz"[:dim])
    ini = _ini(dim, cells, 6, compartments=f"domain.expression = {r2} < 0.2", rk="Alexander2")
    over = (f"model.time_step_operator.linear_solver.precision = {precision}\n"
            f"model.time_step_operator.linear_solver.preconditioner.type = {precond}\n")
    gpu = dca.Model(ini, over, 0, runtime_parameters=runtime)
    orc = OracleModel(ini)
    u0 = gpu.initial_state()
    gpu.set_state(u0, 0.0)
    orc.set_state(u0, 0.0)
    gpu.profile_enable(True)
    t = 0.0
    for _ in range(2):
        st = gpu.step(t, 0.1)
        rc, newton, _ = orc.step(0.1)
        assert st.status == 0 and rc == 0 and st.newton_iterations == newton
        t += 0.1
    assert gpu.profile("point_setup")[0] > 0 and gpu.profile("assembly_jacobian")[0] == 0
    u, _ = gpu.get_state()
    uo, _ = orc.get_state()
    assert max(rel_l2_per_species(gpu.compartments(), u, uo)) < 1e-8
    gpu.close()
    orc.close()


@pytest.mark.parametrize("precond", ["Jacobi", "VertexBlockJacobi"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim,cells", [(2, (66, 40)), (3, (9, 8, 17))])
def test_steps_every_shape(dca, dim, cells, precision, precond):
    """Steps with each tile shape forced, several tiles and remainders along every axis."""
    print(f"case: corner form, every shape, {dim}D {precision} {precond}", flush=True)
    ini = _ini(dim, cells, 6, rk="Alexander2")
    orc = OracleModel(ini)
    u0 = np.random.default_rng(4).random(orc.n_dof) * 0.2 + 0.5
    orc.set_state(u0, 0.0)
    assert orc.step(0.1)[0] == 0
    for tile in (0, 1):
        gpu = dca.Model(ini, f"model.time_step_operator.linear_solver.precision = {precision}\n"
                             f"model.time_step_operator.linear_solver.preconditioner.type = {precond}\n"
                             f"model.time_step_operator.linear_solver.point_tile = {tile}\n", 0)
        assert "dcg_tile_0_e0" in gpu.generated_source()
        gpu.set_state(u0, 0.0)
        assert gpu.step(0.0, 0.1).status == 0
        assert max(rel_l2_per_species(gpu.compartments(), gpu.get_state()[0], orc.get_state()[0])) < 1e-8, tile
        gpu.close()
    orc.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_of_sizes(dca, precision):
    """Members of one module with other sizes, spacings and constants, and one of another block size."""
    print(f"case: corner form batch {precision}", flush=True)
    inis = [_ini(3, (5, 6, 4), 5), _ini(3, (9, 7, 11), 5, extensions=(0.5, 1.0, 1.3)).replace("0.7", "0.9"),
            _ini(2, (40, 35), 7)]
    batch = dca.Batch(f"precision = {precision}\n", 0)
    members, oracles = [], []
    for ini in inis:
        i = batch.add(ini)
        batch.set_time_step(i, 0.1)
        m = batch.member(i)
        o = OracleModel(ini)
        u0 = o.get_state()[0] * 0 + 0.5 + 0.2 * np.random.default_rng(i).random(m.n_dof)
        m.set_state(u0, 0.0)
        o.set_state(u0, 0.0)
        members.append(m)
        oracles.append(o)
    for _ in range(2):
        assert all(s.status == 0 for s in batch.step())
        for o in oracles:
            assert o.step(0.1)[0] == 0
    for m, o in zip(members, oracles):
        assert max(rel_l2_per_species(m.compartments(), m.get_state()[0], o.get_state()[0])) < 1e-8
