"""How the tile blocks are dealt to the XCDs changes no result: a domain large
enough to be dealt in short runs against the same flow on half of it (dealt as
one stretch per XCD), and a batch whose grid crosses the line of its rule
against its members stepped alone."""
import numpy as np
import pytest

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,dims", [("f16", (272, 256, 272)), ("f32", (272, 256, 256))])
def test_large_periodic_box_equals_its_half(storage, dims):
    """The flow has period nz/2 along z, so both halves of the large box and
    the half box hold the same cells with the same neighbours: equal bits.
    D3Q27 f16: 1.02 GB against the line at 1.0; f32: 1.92 against 1.85."""
    import lbmflow_amd as L

    nx, ny, nz = dims
    half = (nx, ny, nz // 2)
    rho, u = cases.tgv_field(half, 0.03)
    got = []
    for d in (half, dims):
        s = L.Solver(27, d, nu=0.01, collision="cm", storage=storage, periodic=(True, True, True))
        k = d[2] // half[2]
        s.init_with(np.tile(rho, k), np.tile(u, (k, 1)))
        s.run(3)
        got.append(np.stack(s.moments()))
        s.close()
    n = nx * ny * half[2]
    assert np.array_equal(got[1][:, :n], got[0])
    assert np.array_equal(got[1][:, n:], got[0])


@pytest.mark.parametrize("grid", [1, 16383, 16384, 16391])
def test_batch_grid_changes_no_result(grid):
    import lbmflow_amd as L

    def make():
        out = []
        for n in (30, 41):
            tc = cases.tank_case(n, nu=0.02, collision="trt", Q=19)
            s = L.Solver(19, (n,) * 3, nu=0.02, collision="trt", solid=tc["solid"])
            s.set_rotating_body(tc["pos"], tc["w"], tc["c"], (0.0, 0.0, tc["omega"]))
            out.append(s)
        return out

    alone, members = make(), make()
    want = [s.run_with_ibm(7)[0] for s in alone]
    b = L.Batch(members)
    b.set_grid(grid)
    tq = b.run(7)
    for k, (a, m) in enumerate(zip(alone, members)):
        assert np.array_equal(tq[k], want[k])
        assert np.array_equal(a.populations(), m.populations())
    b.close()
