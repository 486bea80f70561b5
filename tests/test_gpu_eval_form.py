"""Coefficients evaluated inside the apply (blocks of 1 to 4 species on box
cells) and BiCGSTAB on fused operator launches, against the oracle: Jacobian
apply and steps at sides around the tiles' 3, 4, 7, 15 and 31 vertices, odd
sizes, non-square boxes, a compartment that covers a part of the grid,
interface and boundary terms (rows with facets of several kinds), both Jacobi
forms, FP64 and mixed; and models that keep stored coefficients because one
compartment's expressions cost more than reading them.  Sums run in another
order than the oracle's in FP64: 1e-12 relative for one application, the
parity bar of 1e-8 for converged steps."""
import numpy as np
import pytest

from tests.oracle_lib import OracleModel, rel_l2_per_species

pytestmark = pytest.mark.gpu

PTS = ("model.time_step_operator.linear_solver.storage = points\n"
       "model.time_step_operator.linear_solver.preconditioner.type = {}\n"
       "model.time_step_operator.linear_solver.precision = {}\n")

# far more operations than coefficients: such a compartment stores them
COSTLY = "1e-30*(" + "+".join(f"sin({k}*position_x)*cos({k}+time)" for k in range(1, 24)) + ")"


def _ini(dim, cells, species, inner=0, costly=False, extensions=(1.0, 0.6, 1.7)):
    """`species` species outside a ball, `inner` species inside it with a flux between the first ones (0: no ball)."""
    r2 = " + ".join(f"(position_{a}-0.4)^2" for a in "xyz"[:dim])
    comps = "domain.expression = 1" if not inner else f"domain.expression = {r2} >= 0.08\ncore.expression = {r2} < 0.08"
    out = [f"[grid]\ndimension = {dim}\ncells = {' '.join(map(str, cells))}\n"
           f"extensions = {' '.join(map(str, extensions[:dim]))}\ncell_type = cube", f"[compartments]\n{comps}"]
    for comp, tag, n in (("domain", "s", species), ("core", "c", inner)):
        for i in range(n):
            a, b = f"{tag}{i}", f"{tag}{(i + 1) % n}"
            extra = f" + {COSTLY}" if costly and comp == "domain" and i == 0 else ""
            out += [f"[model.scalar_field.{a}]", f"compartment = {comp}", f"storage.expression = {1.0 + 0.1 * i}",
                    f"initial.expression = 0.5 + 0.1*sin({i + 1}*position_x + 2*position_y)",
                    f"cross_diffusion.{a}.expression = {0.001 * (i + 1)}"]
            if n > 1:
                out += [f"reaction.expression = 0.7*{b}*{b} - {a}*{b} + 0.1*position_x*{a} + 0.05*time*{b}",
                        f"reaction.jacobian.{a}.expression = -{b} + 0.1*position_x{extra}",
                        f"reaction.jacobian.{b}.expression = 1.4*{b} - {a} + 0.05*time"]
            else:
                out += [f"reaction.expression = 0.7*{a}*{a} - 0.05*time*{a}",
                        f"reaction.jacobian.{a}.expression = 1.4*{a} - 0.05*time{extra}"]
            if i == 0 and inner:
                other, sign = ("core", "") if comp == "domain" else ("domain", "-")
                out += [f"outflow.{other}.expression = {sign}0.3*(s0 - c0*c0)",
                        f"outflow.{other}.jacobian.s0.expression = {sign}0.3",
                        f"outflow.{other}.jacobian.c0.expression = {sign}(-0.6*c0)"]
                if comp == "domain":  # the domain's boundary
                    out += ["outflow.domain.expression = 0.2*s0*s0", "outflow.domain.jacobian.s0.expression = 0.4*s0"]
    return "\n".join(out) + ("\n[model.time_step_operator]\ntype = Alexander2\nlinear_solver.type = BiCGSTAB\n"
                             "linear_solver.convergence_condition.relative_tolerance = 1e-12\n"
                             "linear_solver.convergence_condition.iteration_range = 1 2000\n"
                             "linear_solver.preconditioner.type = Jacobi\n"
                             "nonlinear_solver.convergence_condition.relative_tolerance = 1e-20\n"
                             "nonlinear_solver.convergence_condition.absolute_tolerance = 1e-28\n"
                             "nonlinear_solver.convergence_condition.iteration_range = 0 40\n")


SHAPES = [(2, (1, 1)), (2, (7, 4)), (2, (15, 14)), (2, (30, 16)), (2, (47, 33)), (3, (1, 1, 1)), (3, (3, 4, 7)),
          (3, (7, 8, 6)), (3, (8, 3, 15)), (3, (16, 5, 9)), (3, (13, 6, 18)), (3, (28, 14, 34))]


@pytest.mark.parametrize("species", [1, 2, 3, 4])
@pytest.mark.parametrize("dim,cells", SHAPES)
def test_apply(dca, dim, cells, species):
    print(f"case: evaluated form {dim}D {cells} {species} species", flush=True)
    ini = _ini(dim, cells, species)
    orc = OracleModel(ini)
    rng = np.random.default_rng(species)
    x = v = None
    for tile in range(8):
        over = f"model.time_step_operator.linear_solver.point_tile = {tile}\n"
        gpu = dca.Model(ini, PTS.format("Jacobi", "fp64") + over, 0)
        assert "dcg_tile_0_e0" in gpu.generated_source()
        if x is None:
            x, v = 0.5 + 0.2 * rng.random(gpu.n_dof), rng.standard_normal(gpu.n_dof)
        for cm, ca in ((1.0, 0.0), (1.0, 0.3)):
            _, vals = orc.assemble(x, 0.4, cm, ca)
            ref = orc.csr(vals) @ v
            y = gpu.jacobian_apply(x, 0.4, cm, ca, v)
            assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), tile
        gpu.close()
    orc.close()


@pytest.mark.parametrize("costly", [False, True])
@pytest.mark.parametrize("precond", ["Jacobi", "VertexBlockJacobi"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim,cells,species,inner", [(2, (33, 20), 3, 2), (2, (17, 31), 1, 4), (3, (9, 8, 6), 2, 1),
                                                     (3, (8, 7, 11), 4, 6)])
def test_steps(dca, dim, cells, species, inner, precision, precond, costly):
    print(f"case: evaluated form steps {dim}D {species}+{inner} {precision} {precond} costly={costly}", flush=True)
    ini = _ini(dim, cells, species, inner, costly)
    gpu = dca.Model(ini, PTS.format(precond, precision), 0)
    assert ("dcg_tile_0_e0" in gpu.generated_source()) != costly
    orc = OracleModel(ini)
    u0 = gpu.initial_state()
    gpu.set_state(u0, 0.0)
    orc.set_state(u0, 0.0)
    t = 0.0
    for _ in range(2):
        st = gpu.step(t, 0.1)
        rc, newton, _ = orc.step(0.1)
        assert st.status == 0 and rc == 0 and st.newton_iterations == newton
        t += 0.1
    assert max(rel_l2_per_species(gpu.compartments(), gpu.get_state()[0], orc.get_state()[0])) < 1e-8
    gpu.close()
    orc.close()


@pytest.mark.parametrize("precond", ["Jacobi", "VertexBlockJacobi"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("species,inner", [(2, 0), (3, 2), (1, 4)])
def test_steps_every_shape(dca, species, inner, precision, precond):
    """Steps with each tile shape forced, the walked layers among them: several chunks of layers along z and tiles along
    x and y with remainders, partial compartments of other block sizes and facet rows, in both precisions."""
    print(f"case: evaluated form, every shape, {species}+{inner} {precision} {precond}", flush=True)
    ini = _ini(3, (28, 14, 34), species, inner, extensions=(1.0, 1.0, 1.0))
    orc = OracleModel(ini)
    u0 = np.random.default_rng(3).random(orc.n_dof) * 0.2 + 0.5
    orc.set_state(u0, 0.0)
    assert orc.step(0.1)[0] == 0
    ref = orc.get_state()[0]
    walked = 0
    for tile in range(7):
        over = f"model.time_step_operator.linear_solver.point_tile = {tile}\n"
        gpu = dca.Model(ini, PTS.format(precond, precision) + over, 0)
        src = gpu.generated_source()
        assert "dcg_tile_0_e0" in src
        walked += f"_e{tile}, double, vol0::ApplyShape{tile}, eval_march" in src
        gpu.set_state(u0, 0.0)
        assert gpu.step(0.0, 0.1).status == 0
        assert max(rel_l2_per_species(gpu.compartments(), gpu.get_state()[0], ref)) < 1e-8, tile
        gpu.close()
    assert walked == 3
    orc.close()


@pytest.mark.parametrize("inner,precision", [(0, "fp64"), (1, "mixed")])
def test_finished_reductions(dca, inner, precision):
    """1451^2 vertices: more than 2,048 partials of both operators and of the x and r update (1,024 vertices each), so
    that every reduction goes through the finishing launch.  The matrix form of the same step is the reference."""
    print(f"case: evaluated form, finished reductions, inner={inner} {precision}", flush=True)
    ini = _ini(2, (1450, 1450), 1, inner, extensions=(1.0, 1.0, 1.0))
    states = []
    for storage in ("points", "matrix"):
        m = dca.Model(ini, PTS.format("Jacobi", precision).replace("points", storage), 0)
        assert ("dcg_tile_0_e0" in m.generated_source()) == (storage == "points")
        m.set_state(m.initial_state(), 0.0)
        assert m.step(0.0, 0.1).status == 0
        states.append(m.get_state()[0])
        comps = m.compartments()
        m.close()
    assert max(rel_l2_per_species(comps, *states)) < 1e-8


@pytest.mark.parametrize("cells", [(361, 361), (362, 362)])
def test_step_slots_per_thread(dca, cells):
    """Meshes just below and above the 131,072 vertices where the x and r update takes four slots per thread."""
    print(f"case: evaluated form slots {cells}", flush=True)
    ini = _ini(2, cells, 1)
    gpu, orc = dca.Model(ini, PTS.format("Jacobi", "fp64"), 0), OracleModel(ini)
    u0 = gpu.initial_state()
    gpu.set_state(u0, 0.0)
    orc.set_state(u0, 0.0)
    assert gpu.step(0.0, 0.1).status == 0 and orc.step(0.1)[0] == 0
    assert max(rel_l2_per_species(gpu.compartments(), gpu.get_state()[0], orc.get_state()[0])) < 1e-8
    gpu.close()
    orc.close()


@pytest.mark.parametrize("graph", [0, 3, 4])
@pytest.mark.parametrize("precision,precond", [("fp64", "Jacobi"), ("mixed", "Jacobi"), ("fp64", "VertexBlockJacobi"),
                                               ("mixed", "None")])
def test_batch(dca, precision, precond, graph):
    """Members of several modules, sizes and block sizes (one with stored coefficients) on fused iterations, as
    plain launches and captured in odd and even numbers."""
    print(f"case: evaluated form batch {precision} {precond} graph_iterations={graph}", flush=True)
    inis = [_ini(2, (33, 20), 2), _ini(2, (7, 50), 2, extensions=(0.5, 2.0, 1.0)), _ini(2, (16, 9), 2, costly=True),
            _ini(3, (9, 8, 6), 3), _ini(2, (1, 1), 4), _ini(3, (4, 5, 7), 6)]
    batch = dca.Batch(f"precision = {precision}\npreconditioner = {precond}\ngraph_iterations = {graph}\n"
                      "iteration_limit = 2000\n", 0)
    members, oracles = [], []
    for ini in inis:
        i = batch.add(ini)
        batch.set_time_step(i, 0.1)
        m, o = batch.member(i), OracleModel(ini)
        u0 = 0.5 + 0.2 * np.random.default_rng(i).random(m.n_dof)
        m.set_state(u0, 0.0)
        o.set_state(u0, 0.0)
        members.append(m)
        oracles.append(o)
    for _ in range(3):
        assert all(s.status == 0 for s in batch.step())
        for o in oracles:
            assert o.step(0.1)[0] == 0
        for m, o in zip(members, oracles):
            assert max(rel_l2_per_species(m.compartments(), m.get_state()[0], o.get_state()[0])) < 1e-8


def test_compartments_share_scalars(dca):
    """Two compartments whose forced tiles have 256 and 512 threads, about 400 partials: every launch of an iteration
    works with one set of scalars.  The initial state makes r.(J r) cancel to 1e-6 of its terms, so alpha is 1e6 with a
    relative rounding of about 1e-10: compartments with an alpha each leave parts of the right-hand side unsolved (4e-6
    where it happened); with one alpha the true residual is the recursion's (1e-8) up to 1e6 roundings: 1e-7.  The
    state comes from a linear step, which has no later defect test."""
    print("case: evaluated form, scalars of two compartments", flush=True)
    n, off = 40, 41 * 41 * 21 * 4
    out = [f"[grid]\ndimension = 3\ncells = {n} {n} {n}\nextensions = 1 1 1\ncell_type = cube",
           "[compartments]\nlow.expression = position_z < 0.5\nhigh.expression = position_z >= 0.5"]
    for comp, names in (("low", ["a0", "a1", "a2", "a3"]), ("high", ["b0", "b1"])):
        for i, s in enumerate(names):
            jac = {s: "-1"}
            if i % 2 == 0:
                jac[names[i + 1]] = "8"
            if comp == "low":  # a full block, so that the compartments' candidate tiles differ
                jac.update({o: "1e-30" for o in names if o not in jac})
            out += [f"[model.scalar_field.{s}]", f"compartment = {comp}", "storage.expression = 1",
                    "reaction.expression = " + " + ".join(f"{c}*{o}" for o, c in jac.items())]
            out += [f"reaction.jacobian.{o}.expression = {c}" for o, c in jac.items()]
    ini = "\n".join(out) + ("\n[model]\nis_linear = true\n[model.time_step_operator]\ntype = ImplicitEuler\n"
                            "linear_solver.type = BiCGSTAB\n"
                            "linear_solver.convergence_condition.relative_tolerance = 1e-8\n"
                            "linear_solver.convergence_condition.iteration_range = 1 500\n"
                            "linear_solver.preconditioner.type = None\n")
    orc = OracleModel(ini)
    _, vals = orc.assemble(np.zeros(orc.n_dof), 1.0, 1.0, 1.0)
    A = orc.csr(vals)
    x = [np.tile(np.arange(n + 1) / n, 41 * 21) for _ in range(2)]

    def state(inside, sign):  # whose reaction is (1, sign) per pair of species at the vertices inside, else 0
        u = np.zeros(orc.n_dof)
        for part, xs, b in ((u[:off], x[0], 4), (u[off:], x[1], 2)):
            g = inside(xs)[:, None]
            part.reshape(-1, b)[:, 1::2] = -sign * g
            part.reshape(-1, b)[:, 0::2] = -(8 * sign + 1) * g
        return u

    P, Q = state(lambda s: 1.0 * (s < 0.75), 1.0), state(lambda s: 1.0 * (s >= 0.75), -1.0)
    rP, rQ = orc.assemble(P, 1.0, 0.0, 1.0)[0], orc.assemble(Q, 1.0, 0.0, 1.0)[0]
    pp, pq, qq = rP @ (A @ rP), rP @ (A @ rQ) + rQ @ (A @ rP), rQ @ (A @ rQ)
    assert pp < 0 < qq
    a = max(np.roots([qq, pq, pp - 1e-6 * (qq - pp)]).real)
    b = rP + a * rQ
    gpu = dca.Model(ini, PTS.format("None", "fp64") + "model.time_step_operator.linear_solver.point_tile = 2\n", 0)
    src = gpu.generated_source()
    assert "ApplyShape2 = ApplyTile<7, 7, 3, 256" in src and "ApplyShape2 = ApplyTile<7, 7, 7, 512" in src
    gpu.set_state(P + a * Q, 0.0)
    st = gpu.step(0.0, 1.0)
    assert st.status == 0
    z = P + a * Q - gpu.get_state()[0]
    assert np.linalg.norm(b - A @ z) <= 1e-7 * np.linalg.norm(b)
    gpu.close()
    orc.close()


@pytest.mark.parametrize("graph", [0, 4])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_finished_reductions(dca, precision, graph):
    """A 513^2 member in tiles of 16 x 8 rows (2,145 of them) takes its group's reductions through launches of their own;
    members of other sizes and modules in the same group.  Each member's own steps are the reference."""
    print(f"case: evaluated form batch, finished reductions {precision} graph_iterations={graph}", flush=True)
    inis = [_ini(2, (512, 512), 2), _ini(2, (300, 200), 2, extensions=(0.5, 2.0, 1.0)), _ini(2, (9, 7), 2),
            _ini(3, (12, 9, 7), 2)]
    batch = dca.Batch(f"precision = {precision}\npreconditioner = Jacobi\ngraph_iterations = {graph}\n"
                      "iteration_limit = 2000\npoint_tile = 0\n", 0)
    members, singles = [], []
    for ini in inis:
        i = batch.add(ini)
        batch.set_time_step(i, 0.1)
        m, s = batch.member(i), dca.Model(ini, PTS.format("Jacobi", precision), 0)
        u0 = 0.5 + 0.2 * np.random.default_rng(i).random(m.n_dof)
        for x in (m, s):
            x.set_state(u0, 0.0)
        members.append(m)
        singles.append(s)
    for k in range(2):
        assert all(st.status == 0 for st in batch.step())
        for m, s in zip(members, singles):
            assert s.step(0.1 * k, 0.1).status == 0
            assert max(rel_l2_per_species(m.compartments(), m.get_state()[0], s.get_state()[0])) < 1e-8
    for s in singles:
        s.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cells,species,inner", [(n, b, 0) for n in (1, 2, 126, 127, 128, 300) for b in (1, 2, 4)] +
                         [(n, b, i) for n in (126, 127, 128, 300) for b, i in ((3, 2), (1, 4))])
def test_one_dimension(dca, cells, species, inner, precision):
    """Intervals around the tile's 128 vertices: the apply and a step, with an interface where two compartments fit."""
    print(f"case: evaluated form 1D {cells} {species}+{inner} {precision}", flush=True)
    ini = _ini(1, (cells,), species, inner)
    gpu, orc = dca.Model(ini, PTS.format("Jacobi", precision), 0), OracleModel(ini)
    assert "dcg_tile_0_e0" in gpu.generated_source()
    rng = np.random.default_rng(cells)
    x, v = 0.5 + 0.2 * rng.random(gpu.n_dof), rng.standard_normal(gpu.n_dof)
    _, vals = orc.assemble(x, 0.4, 1.0, 0.3)
    ref = orc.csr(vals) @ v
    assert np.abs(gpu.jacobian_apply(x, 0.4, 1.0, 0.3, v) - ref).max() <= 1e-12 * np.abs(ref).max()
    for m in (gpu, orc):
        m.set_state(x, 0.0)
    assert gpu.step(0.0, 0.1).status == 0 and orc.step(0.1)[0] == 0
    assert max(rel_l2_per_species(gpu.compartments(), gpu.get_state()[0], orc.get_state()[0])) < 1e-8
    gpu.close()
    orc.close()
