"""Read-back in pieces through pinned slots: every size class (one slot, one
piece over several slots, several pieces with a ragged last one) returns the
device's values bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 4 N floats against the 2 MiB slot and the 64 MiB workspace (4,194,304 cells
# a piece of moments; Q planes of 862,208 (19) / 620,544 (27) cells of
# populations)
@pytest.mark.parametrize("Q,dims", [(19, (7, 5, 3)), (27, (32, 64, 64)), (19, (33, 64, 64)), (19, (163, 161, 161)),
                                    (27, (97, 81, 79))])
def test_moments_and_populations_in_pieces(Q, dims):
    import lbmflow_amd as L

    n = dims[0] * dims[1] * dims[2]
    rng = np.random.RandomState(5)
    f = (rng.rand(Q, n).astype(np.float32) - np.float32(0.5)) * np.float32(1e-2)
    solid = (rng.rand(n) < 0.1).astype(np.uint8)
    s = L.Solver(Q, dims, nu=0.05, collision="trt", periodic=(True, True, True), solid=solid)
    s.set_populations(f)
    got = s.populations()
    want = np.where(solid[None], np.float32(0.0), f)
    assert np.array_equal(got, want)
    rho, ux, uy, uz = s.moments()
    dr = np.zeros(n, np.float32)
    for q in range(Q):
        dr = dr + f[q]
    assert np.array_equal(rho, np.where(solid, np.float32(1.0), np.float32(1.0) + dr))
    # c_q . f of the axis directions and pairs, f64: fp32 sums of Q terms
    c = np.array([(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0),
                  (-1, -1, 0), (1, 0, 1), (-1, 0, -1), (0, 1, 1), (0, -1, -1), (1, -1, 0), (-1, 1, 0), (1, 0, -1),
                  (-1, 0, 1), (0, 1, -1), (0, -1, 1), (1, 1, 1), (-1, -1, -1), (1, 1, -1), (-1, -1, 1), (1, -1, 1),
                  (-1, 1, -1), (1, -1, -1), (-1, 1, 1)], np.float64)[:Q]
    for a, u in enumerate((ux, uy, uz)):
        ref = np.where(solid, 0.0, c[:, a] @ f.astype(np.float64)) / rho.astype(np.float64)
        # each of at most Q roundings is below 2^-24 of the partial sums' bound Q * 5e-3
        assert np.abs(u - ref).max() <= 2.0 * Q * 2.0 ** -24 * Q * 5e-3
    s.close()


def test_small_domain_holds_little_device_memory():
    """Reads of a 16^3 domain keep what they need, not the workspace's bound."""
    import ctypes as C

    import lbmflow_amd as L

    ctx = L.Context(0)

    def free_bytes():  # by the runtime the library is linked with
        f, t = C.c_size_t(), C.c_size_t()
        assert ctx.lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    s = L.Solver(19, (16, 16, 16), nu=0.05, periodic=(True,) * 3, ctx=ctx)
    s.run(2)
    before = free_bytes()
    s.moments()
    s.populations()
    assert before - free_bytes() <= 8 << 20
    s.close()


def test_a_context_closed_first_serves_its_domains():
    """At interpreter exit a context can be finalized before the solvers and
    batches on it: they keep what they use of it until the last of them goes."""
    import lbmflow_amd as L

    ctx = L.Context(0)
    s = []
    for n in (12, 14):
        s.append(L.Solver(19, (n,) * 3, nu=0.05, ctx=ctx))
        s[-1].build_wall_rims([1] * 6, np.eye(6, 3) * 0.02)
    b = L.Batch(s)
    ctx.close()
    b.run(2)
    rho = s[0].moments()[0]
    assert np.all(np.isfinite(rho)) and s[1].time == 2
    s[0].close()
    b.close()
    s[1].run(1)
    assert s[1].populations().shape == (19, 14 ** 3)
    s[1].close()
