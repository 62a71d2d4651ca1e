"""The WALE closure inside the collide-stream kernel (closed domains) against
the closure's own update before each step, over what both accept: lattices,
collisions, storages, moving walls, a clip, force-listed cells, both parities.

Both forms run the same operations in the same order: equal bits."""
import numpy as np
import pytest

import lbmflow_amd as L
from oracle import oracle as O
from tests import cases

pytestmark = pytest.mark.gpu


def cavity(Q, collision, storage, dims, lid=0.08):
    u = np.zeros((6, 3))
    u[5] = [lid, 0.0, 0.0]
    s = L.Solver(Q, dims, nu=0.004, collision=collision, storage=storage)
    s.build_wall_rims([1] * 6, u)
    solid = s.solid().reshape(dims[2], dims[1], dims[0])
    solid[4:6, 3:5, 5:8] = 1  # an obstacle: walls on either side, one-cell gaps
    solid[4:6, 3:5, 9] = 1
    wall = np.zeros((*solid.shape, 3), np.float32)
    wall[-1, :, :, 0] = lid
    s.set_masks(solid.reshape(-1), wall.reshape(-1))
    rho, uu = cases.tgv_field(dims, 0.03)
    s.init_with(rho, uu)
    return s, solid.reshape(-1) == 0


@pytest.mark.parametrize("dims", [(64, 12, 11), (19, 13, 9)])  # row tiles and linear tiles
@pytest.mark.parametrize("Q,collision,storage", [(19, "trt", "f32"), (27, "trt", "f32"), (27, "cm", "f32"),
                                                 (19, "cm", "f32"), (27, "cm", "f16"), (19, "bgk", "bf16")])
@pytest.mark.parametrize("clip", [False, True])
def test_closure_inside_equals_update_before_each_step(Q, collision, storage, dims, clip):
    tau = 0.5 + 3 * 0.004 + 3e-4 if clip else None
    a, fl = cavity(Q, collision, storage, dims)
    b, _ = cavity(Q, collision, storage, dims)
    a.set_wale(True, tau_eff_max=tau)
    for _ in range(5):
        b.wale_update(tau_eff_max=tau)
        want = b.omega_field()
        b.run(1)
        a.run(1)
        got = a.omega_field()
        assert np.array_equal(got, want)
    assert np.array_equal(a.populations(), b.populations())
    a.close()
    b.close()


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_body_and_riding_scalar(storage):
    """A tank with a rotating body, the closure and a D3Q7 tracer whose step
    rides on the next step's velocity pass: spans of any length, captured or
    not, equal one step at a time bit for bit; a force field off the body too."""
    tc = cases.tank_case(28, nu=0.004)
    outs = []
    for mode in ("single", "eager", "graph"):
        s = L.Solver(27, (28,) * 3, nu=0.004, collision="cm", storage=storage, solid=tc["solid"])
        s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
        k = s.enable_scalar_distribution(0.01, "d3q7")
        s.set_scalar_concentration(k, tc["blob"])
        s.set_wale(True)
        out = []
        for n in (1, 6, 5, 2, 3):
            if mode == "single":
                tq = np.concatenate([s.run_with_ibm(1, graph=False)[0] for _ in range(n)])
            else:
                tq, _ = s.run_with_ibm(n, graph=mode == "graph")
            out += [tq, s.gather_scalar_concentration(k), s.omega_field(), np.stack(s.moments())]
        s.set_wale(False)
        s.run_with_ibm(3, graph=mode == "graph")
        out += [s.gather_scalar_concentration(k), s.populations()]
        outs.append(out)
        s.close()
    for o in outs[1:]:
        for x, y in zip(outs[0], o):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("storage,dims,steps", [("f32", (64, 12, 11), 3), ("f16", (19, 13, 9), 2)])
def test_tiles_autotuned_under_the_closure_leave_the_field(storage, dims, steps):
    s, fl = cavity(27, "cm", storage, dims)
    b, _ = cavity(27, "cm", storage, dims)
    for v in (s, b):
        v.set_wale(True)
        v.run(steps)
    om, f = s.omega_field(), s.populations()
    s.autotune_tiles(4)
    assert np.array_equal(s.omega_field(), om) and np.array_equal(s.populations(), f)
    for v in (s, b):
        v.run(3)
    assert np.array_equal(s.omega_field(), b.omega_field()) and np.array_equal(s.populations(), b.populations())
    s.close()
    b.close()


def test_calls_without_a_step_leave_the_field():
    """After the closure is switched on (again) the installed field stands until
    a step writes it: spans of no step and the autotuner leave it alone."""
    tc = cases.tank_case(28, nu=0.004)
    s = L.Solver(27, (28,) * 3, nu=0.004, collision="cm", solid=tc["solid"])
    s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
    s.set_wale(True)
    s.run_with_ibm(3)
    computed = s.omega_field()
    given = (1.0 + 0.2 * np.random.RandomState(1).rand(s.n)).astype(np.float32)
    for field in (computed, given):
        s.set_omega_field(field)
        s.set_wale(True)
        for call in (lambda: s.run(0), lambda: s.run_with_ibm(0), lambda: s.autotune_tiles(4)):
            call()
            assert np.array_equal(s.omega_field(), field)
    s.set_wale(False)
    assert np.array_equal(s.omega_field(), given)
    # and a step writes all of it, the solid cells included
    s.set_wale(True)
    s.run_with_ibm(1)
    solid = tc["solid"].reshape(-1) != 0
    rate = np.float32(1.0) / (np.float32(3.0) * np.float32(0.004) + np.float32(0.5))
    assert np.abs(s.omega_field()[solid] - rate).max() <= 2.0 ** -21  # last bits of the sum (2^-24) and of a quotient near 2
    assert not np.array_equal(s.omega_field()[~solid], given[~solid])
    s.close()


@pytest.mark.parametrize("Q,collision", [(27, "cm"), (19, "trt")])
def test_tank_with_body_follows_the_oracle(Q, collision):
    tc = cases.tank_case(30, collision=collision, Q=Q, nu=0.004)
    steps = 6
    s = L.Solver(Q, (30,) * 3, nu=tc["nu"], collision=collision, solid=tc["solid"])
    s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
    s.set_wale(True)
    s.run_with_ibm(steps)
    o = O.OracleSolver(Q, (30,) * 3, prec=4, collision=cases.COLL[collision], nu=tc["nu"], solid=tc["solid"])
    for _ in range(steps):
        o.clear_force_field()
        o.apply_ibm(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
        om, _, _, _ = o.wale()
        o.set_omega_field(om)
        o.step(1)
    fl = tc["solid"] == 0
    assert np.abs(s.populations()[:, fl].astype(np.float64) - o.get_f()[:, fl]).max() < 2e-6
    s.close()


@pytest.mark.parametrize("kind", ["closed", "periodic", "tracer"])
@pytest.mark.parametrize("Q,collision,storage", [(27, "cm", "f32"), (19, "trt", "f32"), (27, "trt", "f16"),
                                                 (19, "bgk", "bf16")])
def test_loads_of_the_velocity_pass_give_the_same_bits(kind, Q, collision, storage, monkeypatch):
    """The velocity pass with ordinary and with non-temporal population loads,
    both parities: the choice goes by the domain's size."""
    dims = (19, 13, 9)
    out = []
    for nt in ("0", "1"):
        monkeypatch.setenv("LBM_WALE_NT", nt)
        if kind == "periodic":
            solid = np.zeros((9, 13, 19), np.uint8)
            solid[3:5, 4, 6:8] = 1
            s = L.Solver(Q, dims, nu=0.004, collision=collision, storage=storage, periodic=(True,) * 3,
                         solid=solid.reshape(-1))
            s.init_with(*cases.tgv_field(dims, 0.03))
        else:
            s, _ = cavity(Q, collision, storage, dims)
        if kind == "tracer":
            k = s.enable_scalar_distribution(0.01, "d3q7")
            s.set_scalar_concentration(k, np.linspace(0.0, 1.0, s.n, dtype=np.float32))
        s.set_wale(True)
        s.run(1)
        a = [s.omega_field()]
        s.run(4)
        a += [s.omega_field(), s.populations()]
        if kind == "tracer":
            a.append(s.gather_scalar_concentration(k))
        out.append(a)
        s.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
