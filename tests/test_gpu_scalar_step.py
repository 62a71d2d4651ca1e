"""The scalar step on the device against the reference's three passes
(solver.rs:2113-2205) restated in numpy fp32 with the device's own velocities:
collide in place, pull stream with bounce-back, C = sum h.  Bit for bit, over
re-set concentrations, changed masks and captured spans."""
import numpy as np
import pytest

from tests import cases

pytestmark = pytest.mark.gpu

C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
     (1, 0, 1), (-1, 0, -1), (0, 1, 1), (0, -1, -1), (1, -1, 0), (-1, 1, 0), (1, 0, -1), (-1, 0, 1), (0, 1, -1),
     (0, -1, 1), (1, 1, 1), (-1, -1, -1), (1, 1, -1), (-1, -1, 1), (1, -1, 1), (-1, 1, -1), (1, -1, -1), (-1, 1, 1)]
W = {7: (1 / 4, 1 / 8), 19: (1 / 3, 1 / 18, 1 / 36), 27: (8 / 27, 2 / 27, 1 / 54, 1 / 216)}
f4 = np.float32


class Reference:
    """h and C as the three passes leave them; arrays of shape (nz, ny, nx)."""

    def __init__(self, Qs, dims, D):
        self.Qs, self.shape = Qs, (dims[2], dims[1], dims[0])
        self.k = f4(4.0 if Qs == 7 else 3.0)
        self.om = f4(1.0 / ((4.0 if Qs == 7 else 3.0) * D + 0.5))
        self.w = [f4(W[Qs][sum(abs(v) for v in C[q])]) for q in range(Qs)]
        self.h2 = np.zeros((Qs, *self.shape), f4)

    def heq(self, c, u):
        out = []
        for q in range(self.Qs):
            cu = f4(0.0)
            for a in range(3):
                if C[q][a]:
                    cu = cu + (u[a] if C[q][a] > 0 else -u[a])
            out.append(self.w[q] * c * (f4(1.0) + self.k * cu))
        return out

    def set(self, c, u):
        self.c = c.reshape(self.shape).copy()
        self.h = np.stack(self.heq(self.c, u)).astype(f4)

    def step(self, solid, u):
        eq = self.heq(self.c, u)
        for q in range(self.Qs):
            self.h[q] = np.where(solid, self.h[q], self.h[q] - self.om * (self.h[q] - eq[q]))
        new, s = np.zeros_like(self.h), np.zeros(self.shape, f4)
        for q in range(self.Qs):
            o = 0 if q == 0 else (q + 1 if q % 2 else q - 1)
            ax, sh = (0, 1, 2), (C[q][2], C[q][1], C[q][0])
            v = np.where(np.roll(solid, sh, ax), self.h[o], np.roll(self.h[q], sh, ax))
            new[q] = np.where(solid, f4(0.0), v)
            s = s + new[q]
        self.h2, self.h, self.c = self.h, new, s


def velocity(s):
    d = (s.dims[2], s.dims[1], s.dims[0])
    return [v.reshape(d) for v in s.moments()[1:]]


def domain(Q, storage, periodic_x):
    """Walls in y and z (and x unless periodic) around a driven flow."""
    import lbmflow_amd as L

    dims = (23, 12, 10)
    solid = np.zeros((dims[2], dims[1], dims[0]), np.uint8)
    solid[0] = solid[-1] = 1
    solid[:, 0] = solid[:, -1] = 1
    if not periodic_x:
        solid[:, :, 0] = solid[:, :, -1] = 1
    solid[3:5, 4:7, 9:12] = 1
    s = L.Solver(Q, dims, nu=0.05, collision="trt", storage=storage, periodic=(periodic_x, False, False),
                 force=(1e-5, 2e-6, 0.0), solid=solid.reshape(-1))
    rho, u = cases.tgv_field(dims, 0.02)
    s.init_with(rho, u)
    return s, solid.astype(bool)


@pytest.mark.parametrize("periodic_x", [False, True])
@pytest.mark.parametrize("Q,storage,lattice", [(19, "f32", "d3q7"), (19, "f32", "hydro"), (27, "f16", "d3q7"),
                                               (27, "bf16", "hydro")])
def test_scalar_step_equals_three_passes(Q, storage, lattice, periodic_x):
    s, solid = domain(Q, storage, periodic_x)
    k = s.enable_scalar_distribution(0.03, lattice)
    ref = Reference(7 if lattice == "d3q7" else Q, s.dims, 0.03)
    rng = np.random.RandomState(3)

    def put():
        c = rng.rand(s.n).astype(f4)  # solid cells too: the first step clears them
        s.set_scalar_concentration(k, c)
        ref.set(c, velocity(s))

    def go(n):
        for _ in range(n):
            s.step()
            ref.step(solid, velocity(s))
            got = s.gather_scalar_concentration(k).reshape(ref.shape)
            assert np.array_equal(got, ref.c)

    put()
    go(3)
    put()
    go(2)
    # more solid, then less: the masks change between steps
    for box in ((slice(2, 5), slice(2, 5), slice(5, 8)), None):
        new = solid.copy()
        if box is not None:
            new[box] = True
        else:
            new[3:5, 4:7, 9:12] = False
        s.set_masks(new.astype(np.uint8).reshape(-1))
        solid = new
        go(3)
    s.close()


@pytest.mark.parametrize("lattice", ["d3q7", "hydro"])
def test_captured_spans_after_set_and_stage_in(lattice):
    """Odd and even captured spans, a concentration set and populations staged
    in between them, against one step at a time."""
    import lbmflow_amd as L

    tc = cases.tank_case(26, nu=0.02, collision="trt", Q=19)
    runs = []
    for graph in (True, False):
        s = L.Solver(19, (26,) * 3, nu=0.02, collision="trt", solid=tc["solid"])
        s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
        k = s.enable_scalar_distribution(0.02, lattice)
        s.set_scalar_concentration(k, tc["blob"])
        out = []
        for n in (6, 5, 4):
            for _ in range(1 if graph else n):
                s.run_with_ibm(n if graph else 1, graph=graph)
            out.append(s.gather_scalar_concentration(k))
            out.append(np.array(s.scalar_cv(k)))
        s.set_scalar_concentration(k, tc["blob"] * 0.5)
        s.set_populations(s.populations())
        for n in (7, 2):
            for _ in range(1 if graph else n):
                s.run_with_ibm(n if graph else 1, graph=graph)
            out.append(s.gather_scalar_concentration(k))
        runs.append(out)
        s.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
