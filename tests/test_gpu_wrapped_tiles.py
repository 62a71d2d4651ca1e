"""Linear tiles on domains whose offsets wrap (periodic axes, open faces)
against row tiles: the same populations bit for bit, at row lengths on either
side of the rule and at its edge (55 and 111 cells the last to be packed, 56 and
112 the first rows kept), with solids, moving walls and forces.  The wall rows of
the mixed domains hold all-solid half tiles."""
import numpy as np
import pytest

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [9, 55, 56, 65, 70, 100, 111, 112, 120, 201])
@pytest.mark.parametrize("Q,collision,storage,kind", [(19, "trt", "f32", "periodic"), (27, "cm", "f32", "periodic"),
                                                      (27, "trt", "bf16", "periodic"), (27, "cm", "f16", "mixed"),
                                                      (27, "cm", "f32", "mixed"), (27, "trt", "f32", "mixed"),
                                                      (19, "bgk", "f32", "mixed"), (19, "trt", "f32", "open"),
                                                      (27, "trt", "f32", "open")])
def test_linear_tiles_equal_row_tiles(nx, Q, collision, storage, kind, monkeypatch):
    import lbmflow_amd as L

    dims = (nx, 7, 6)
    solid = np.zeros((6, 7, nx), np.uint8)
    wall = np.zeros((6, 7, nx, 3), np.float32)
    per = (True, True, True)
    if kind == "mixed":  # periodic x, walls in y and z, the upper one moving
        per = (True, False, False)
        solid[0] = solid[-1] = 1
        solid[:, 0] = solid[:, -1] = 1
        wall[-1, :, :, 0] = 0.04
    elif kind == "open":
        per = (False, False, True)
        solid[:, 0] = solid[:, -1] = 1
    solid[2:4, 3, nx // 2:nx // 2 + 2] = 1
    rho, u = cases.tgv_field(dims, 0.02)
    got, held = [], []
    for row in ("1", "0"):
        monkeypatch.setenv("LBM_ROW_TILES", row)
        s = L.Solver(Q, dims, nu=0.03, collision=collision, storage=storage, periodic=per,
                     force=(1e-5, 0.0, -2e-6) if kind != "open" else (0.0, 0.0, 0.0), solid=solid.reshape(-1),
                     wall_u=wall.reshape(-1) if kind == "mixed" else None)
        if kind == "open":
            s.set_face_bc("x-", "velocity", (0.03, 0.0, 0.0))
            s.set_face_bc("x+", "pressure", (1.0,))
        s.init_with(rho, u)
        ff = np.zeros((s.n, 3), np.float32)
        ff[5::17, 1] = 1e-5
        if kind != "open":
            s.set_body_force_field(ff)
        out = []
        for n in (1, 2, 4):
            s.run(n)
            out.append(s.populations())
        got.append(out)
        held.append(s.device_bytes())
        s.close()
    nseg = (nx + 63) // 64
    assert (held[0] != held[1]) == (nseg * 64 - nx > nseg * 8)  # packed tiles are fewer
    for a, b in zip(*got):
        assert np.array_equal(a, b)
