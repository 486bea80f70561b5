"""Transform/reduce in two device levels (workgroups of 256 cells, then one
workgroup per key over their partials): cell counts around both levels' edges
(1, 255 to 257 cells, more than 256 x 256 cells), a second compartment, and
more key texts than a model keeps.  Integrals
of 1 and x over the box and the extremes of quadrature points are known in
closed form: sums of up to 90,000 terms, 1e-12 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = """[volume]
evaluation.expression = integration_factor
[moment]
evaluation.expression = u*integration_factor
[highest]
evaluation.expression = position_x
reduction.expression = a, b: max(a, b)
initial.value = -1e100
[lowest]
evaluation.expression = position_x
reduction.expression = a, b: min(a, b)
initial.value = 1e100
"""


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("cells", [(1, 1), (51, 5), (16, 16), (257, 1), (300, 300)])
def test_reduce_levels(dca, cells, split):
    print(f"case: reduce {cells} split={split}", flush=True)
    comps = "domain.expression = 1" if not split else "domain.expression = position_y >= 0\nnone.expression = 0"
    ini = (f"[grid]\ndimension = 2\ncells = {cells[0]} {cells[1]}\nextensions = 2 3\ncell_type = cube\n"
           f"[compartments]\n{comps}\n[model.scalar_field.u]\ncompartment = domain\nstorage.expression = 1\n"
           "cross_diffusion.u.expression = 0.1\ninitial.expression = position_x\n[model.time_step_operator]\n"
           "type = ImplicitEuler\n")
    m = dca.Model(ini, "", 0)
    m.set_state(m.initial_state(), 0.0)
    hx = 2.0 / cells[0]
    edge = 0.5 - 0.5 * np.sqrt(0.6)  # the three-point Gauss rule's distance from a cell's side
    expect = {"volume": 6.0, "moment": 6.0, "highest": 2.0 - edge * hx, "lowest": edge * hx}
    for _ in range(2):
        got = m.reduce(KEYS)
        for k, v in expect.items():
            assert abs(got[k] - v) <= 1e-12 * abs(v), k
    # another state, other texts in between
    u = m.get_state()[0]
    m.set_state(3 * u, 0.0)
    for i in range(6):
        assert abs(m.reduce(f"[v{i}]\nevaluation.expression = {i + 1}*integration_factor\n")[f"v{i}"]
                   - 6.0 * (i + 1)) <= 1e-11
    assert abs(m.reduce(KEYS)["moment"] - 18.0) <= 1e-10
    m.close()


@pytest.mark.parametrize("cells", [(2, 2), (16, 16), (52, 6), (300, 300), (516, 514)])
def test_fold_order(dca, cells):
    """A reduction that keeps the later value returns the last one in the order of cells (by parity of their indices, so
    with even sides the corner cell comes last), whatever level it passes through."""
    print(f"case: reduce order {cells}", flush=True)
    m = dca.Model(f"[grid]\ndimension = 2\ncells = {cells[0]} {cells[1]}\nextensions = 2 3\ncell_type = cube\n"
                  "[compartments]\ndomain.expression = 1\n[model.scalar_field.u]\ncompartment = domain\n"
                  "storage.expression = 1\ncross_diffusion.u.expression = 0.1\ninitial.expression = position_x\n"
                  "[model.time_step_operator]\ntype = ImplicitEuler\n", "", 0)
    m.set_state(m.initial_state(), 0.0)
    got = m.reduce("[last]\nevaluation.expression = position_x + 10*position_y\nreduction.expression = a, b: a\n"
                   "initial.value = 7\n")
    edge = 0.5 - 0.5 * np.sqrt(0.6)
    assert abs(got["last"] - (2 - edge * 2 / cells[0] + 10 * (3 - edge * 3 / cells[1]))) <= 1e-12 * 32
    m.close()


def test_kept_plans_count_as_footprint(dca):
    """A plan holds (value, defined) pairs per key: one per workgroup of 256 cells and one result."""
    print("case: reduce plans in the footprint", flush=True)
    m = dca.Model("[grid]\ndimension = 2\ncells = 100 100\nextensions = 1 1\ncell_type = cube\n[compartments]\n"
                  "domain.expression = 1\n[model.scalar_field.u]\ncompartment = domain\nstorage.expression = 1\n"
                  "cross_diffusion.u.expression = 0.1\ninitial.expression = position_x\n[model.time_step_operator]\n"
                  "type = ImplicitEuler\n", "", 0)
    m.set_state(m.initial_state(), 0.0)
    before = m.device_bytes()
    m.reduce(KEYS)
    plan = 4 * 16 * (-(-100 * 100 // 256) + 1)
    assert m.device_bytes() == before + plan
    for i in range(6):  # four are kept
        m.reduce(f"[v{i}]\nevaluation.expression = {i + 1}*integration_factor\n")
    assert m.device_bytes() == before + 4 * plan // 4
    m.close()
