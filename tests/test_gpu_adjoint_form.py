"""The adjoint collide-stream kernel over the forms it accepts: periodic axes,
BGK, obstacles with walls on every side and forced cells in wall-linked places,
against finite differences of J with respect to the per-cell viscosity (the
test of test_gpu_adjoint at other domains); 16-bit storage against the fp32
gradient from the same state; the largest domains; and what the call leaves
behind."""
import numpy as np
import pytest

import lbmflow_amd as L
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("collision,periodic,dims", [("trt", (1, 0, 0), (21, 15, 13)), ("bgk", (0, 0, 0), (18, 17, 13)),
                                                     ("trt", (1, 1, 1), (16, 12, 9))])
def test_directional_gradient_matches_differences(collision, periodic, dims):
    nx, ny, nz = dims
    solid = np.zeros((nz, ny, nx), np.uint8)
    for ax, p in enumerate(periodic):
        if not p:
            ix = [slice(None)] * 3
            for k in (0, -1):
                ix[2 - ax] = k
                solid[tuple(ix)] = 1
    solid[3:6, 4:6, 5:7] = 1  # beside the body: forced cells carry wall links
    rng = np.random.RandomState(2)
    c = np.array([nx / 2.0, ny / 2.0, nz / 2.0])
    pos = c + rng.uniform(-3.0, 3.0, (30, 3))
    n, steps, window, nu0, om = nx * ny * nz, 24, 9, 0.05, 0.012
    w = 0.3 * np.ones(30)

    def solver(nu):
        s = L.Solver(19, dims, nu=nu0, collision=collision, periodic=periodic, solid=solid.reshape(-1))
        s.set_omega_field((1.0 / (3.0 * nu + 0.5)).astype(np.float32))
        s.set_rotating_body(pos, w, c, (0.0, 0.0, om))
        return s

    def J(nu):
        s = solver(nu)
        v = s.adjoint_torque(steps, window, 0, gradients=False)["J"]
        s.close()
        return v

    nu = np.full(n, nu0)
    s = solver(nu)
    a = s.adjoint_torque(steps, window, 3)
    s.close()
    s = solver(nu)
    b = s.adjoint_torque(steps, window, 24)
    s.close()
    assert a["J"] == b["J"] and np.array_equal(a["dJ_dnu"], b["dJ_dnu"])
    assert np.all(a["dJ_dnu"][solid.reshape(-1) != 0] == 0.0)
    x, y, z = cases.coords(dims)
    d = nu0 * np.cos(2 * np.pi * (x + 2 * y) / nx) * (solid.reshape(-1) == 0)
    eps = 2e-2
    diff = [(J(nu + e * d) - J(nu - e * d)) / (2 * e) for e in (eps, 0.5 * eps)]
    fd = (4.0 * diff[1] - diff[0]) / 3.0  # the second-order error cancels
    ad = float(np.dot(a["dJ_dnu"], d))
    # fp32 forward: J carries about 1e-7 of rounding against steps of 1e-2
    assert abs(ad - fd) <= 2e-3 * abs(fd) + 1e-5 * abs(a["J"])


@pytest.mark.parametrize("storage,eps", [("f16", 2.0 ** -11), ("bf16", 2.0 ** -8)])
@pytest.mark.parametrize("before", [2, 3])  # the state's parity
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 1, 1)])
def test_sixteen_bit_gradient_from_an_exact_state(storage, eps, before, periodic):
    """Two steps from a 16-bit state, and from the same values held in fp32.
    With the torque of the second step alone the viscosity acts in the first,
    whose populations are the same numbers in both, so that the gradients differ
    by how the second step's rounded velocities and densities enter the body's
    update: a few units of the storage's last place."""
    dims = nx, ny, nz = 21, 16, 13
    solid = np.zeros((nz, ny, nx), np.uint8)
    if not periodic[0]:
        for ax in range(3):
            for k in (0, -1):
                ix = [slice(None)] * 3
                ix[ax] = k
                solid[tuple(ix)] = 1
    solid[3:6, 4:6, 5:7] = 1
    rng = np.random.RandomState(7)
    c = np.array([nx / 2.0, ny / 2.0, nz / 2.0])
    pos = c + rng.uniform(-3.0, 3.0, (30, 3))
    nu = 0.05 * (1.0 + 0.2 * rng.rand(nx * ny * nz))
    rho, u = cases.tgv_field(dims, 0.02)

    def solver(st):
        s = L.Solver(19, dims, nu=0.05, collision="trt", storage=st, periodic=periodic, solid=solid.reshape(-1))
        s.set_omega_field((1.0 / (3.0 * nu + 0.5)).astype(np.float32))
        return s

    a, b = solver(storage), solver("f32")
    a.init_with(rho, u)
    a.run(before)
    b.set_populations(a.populations())
    out = []
    for s in (a, b):
        s.set_rotating_body(pos, 0.3 * np.ones(30), c, (0.0, 0.0, 0.012))
        out.append(s.adjoint_torque(2, 1, 2))
        s.close()
    x, y = out
    for k in ("J", "dJ_domega"):
        assert abs(x[k] - y[k]) <= 8 * eps * abs(y[k])
    d = x["dJ_dnu"] - y["dJ_dnu"]
    assert np.linalg.norm(y["dJ_dnu"]) > 0.0 and np.linalg.norm(d) <= 8 * eps * np.linalg.norm(y["dJ_dnu"])


def test_domain_beyond_the_lane_offset_is_refused():
    """An f64 plane of 2^29 cells is 4 GiB, past the reverse kernel's 32-bit
    byte offset: the gradient is refused before anything else is looked at (no
    body is registered here), the forward-only call as before."""
    s = L.Solver(19, (1024, 1024, 512), nu=0.02, storage="f16", periodic=(True,) * 3)
    with pytest.raises(L.LbmError) as e:
        s.adjoint_torque(2, 1, 1)
    assert e.value.code == -2 and "2^29" in str(e.value)
    with pytest.raises(L.LbmError) as e:
        s.adjoint_torque(2, 1, 1, gradients=False)
    assert e.value.code == -5  # no body
    s.close()


def test_large_domain_gives_the_small_domain_gradient():
    """148.6 M cells: the zeroed adjoint arrays hold more than 2^32 doubles.
    What the body of a resting fluid reaches in four steps is the same cells in
    a small domain, so the gradient there has the same bits and is zero
    elsewhere."""
    rng = np.random.RandomState(4)
    c = np.array([32.0, 32.0, 24.0])
    pos = c + rng.uniform(-3.0, 3.0, (20, 3))
    out = []
    for nz in (48, 36272):
        s = L.Solver(19, (64, 64, nz), nu=0.05, storage="f16", periodic=(True,) * 3)
        s.set_rotating_body(pos, 0.3 * np.ones(20), c, (0.0, 0.0, 0.012))
        out.append(s.adjoint_torque(4, 2, 1))
        s.close()
    small, large = out
    n = small["dJ_dnu"].size
    assert 29 * large["dJ_dnu"].size > 2 ** 32
    assert small["J"] == large["J"] != 0.0 and small["dJ_domega"] == large["dJ_domega"] != 0.0
    assert np.any(small["dJ_dnu"] != 0.0)
    assert np.array_equal(large["dJ_dnu"][:n], small["dJ_dnu"]) and not np.any(large["dJ_dnu"][n:])


@pytest.mark.parametrize("snapshots", [0, 3])
def test_gradient_leaves_the_tracers_of_the_forward_steps(snapshots):
    """The steps that the reverse pass takes again do not move the passive
    scalars: the concentrations after the call are those after the same steps
    without it, bit for bit, and so are those of the steps that follow."""
    n, steps = 24, 9
    tc = cases.tank_case(n, nu=0.02, collision="trt", Q=19)

    def solver():
        s = L.Solver(19, (n,) * 3, nu=0.02, collision="trt", solid=tc["solid"])
        s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
        for lat in ("d3q7", "hydro"):
            s.set_scalar_concentration(s.enable_scalar_distribution(0.01, lat), tc["blob"])
        return s

    a, b = solver(), solver()
    res = a.adjoint_torque(steps, 4, snapshots)
    assert res["forward_steps"] > steps
    b.run_with_ibm(steps)
    for k in (0, 1):
        assert np.array_equal(a.gather_scalar_concentration(k), b.gather_scalar_concentration(k))
    for s in (a, b):
        s.run_with_ibm(3)
    for k in (0, 1):
        assert np.array_equal(a.gather_scalar_concentration(k), b.gather_scalar_concentration(k))
    assert a.time == b.time
    a.close()
    b.close()


@pytest.mark.parametrize("snapshots", [0, 3])
def test_gradient_leaves_the_state_of_the_forward_steps(snapshots):
    """Populations, force field, torque integral and probed force after the
    call are those after the same steps without it, bit for bit, also for a
    plain step that still uses the force field."""
    n, steps = 24, 9
    tc = cases.tank_case(n, nu=0.02, collision="trt", Q=19)

    def solver():
        s = L.Solver(19, (n,) * 3, nu=0.02, collision="trt", solid=tc["solid"])
        s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
        s.set_force_probe(tc["solid"])
        return s

    def state(s):
        torque, updates = s.torque_integral()
        return [s.populations(), s.body_force_field(), torque, s.probed_force(), np.array([updates, s.time])]

    a, b = solver(), solver()
    assert a.adjoint_torque(steps, 4, snapshots)["forward_steps"] > steps
    b.run_with_ibm(steps)
    for call in (None, lambda s: s.run(1), lambda s: s.run_with_ibm(2)):
        for s in (a, b):
            if call:
                call(s)
        for x, y in zip(state(a), state(b)):
            assert np.array_equal(x, y)
    a.close()
    b.close()


def test_a_gradient_refused_for_memory_leaves_the_solver_usable():
    """6,000 snapshots of a 96^3 tank do not fit any card: the call says so,
    and the next one is not blamed for it."""
    tc = cases.tank_case(96, nu=0.01, collision="trt", Q=19)
    s = L.Solver(19, (96,) * 3, nu=0.01, collision="trt", solid=tc["solid"])
    s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
    with pytest.raises(L.LbmError) as e:
        s.adjoint_torque(6000, 10, 5999)
    assert e.value.code == -4
    s.run_with_ibm(2)
    assert s.time == 2
    s.close()
