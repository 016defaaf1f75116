"""Triangle stage kernels at the edges of their element tiles on an MI355X,
against the triangle oracle: a mesh smaller than a wave's group of elements,
exactly one tile (32 elements), a tile and a remainder, several tiles.

Bars: the residual's 1e-12 (FP64) and 1e-5 (FP32-bulk), relative L2.  A step's
increment is a few 1e-3 of the state at these time steps, so the state's
rounding (1e-16 FP64) shows in it at 1e-13 and the bar holds for it too; the
FP32-bulk increment carries the residual's own FP32 error.
"""
import numpy as np
import pytest

from oracle import tri_oracle as T
from tests.test_gpu_parity import rel, say
from tests.test_gpu_tri_viscous import _pair, _state
from zhijian_amd import cases
from zhijian_amd.tri import TriSolver, sp_coords, tri_faces

pytestmark = pytest.mark.gpu

BAR = {"fp64": 1e-12, "fp32bulk": 1e-5}


@pytest.mark.parametrize("n", [1, 4, 5, 9])
@pytest.mark.parametrize("p,precision", [(1, "fp64"), (2, "fp64"), (3, "fp64"), (5, "fp64"), (1, "fp32bulk"), (2, "fp32bulk"),
                                         (3, "fp32bulk"), (4, "fp32bulk"), (5, "fp32bulk")])
def test_tri_viscous_tiles(p, precision, n):
    corr = {1: "dg", 4: "ga", 5: "hu", 9: "sd"}[n]
    say(f"case: triangle viscous stage, {2 * n * n} elements P{p} {precision} roe/{corr}")
    s, o, m = _pair(n, p, "roe", corr, precision=precision, seed=n)
    U = _state(m, p, 7 + n)
    s.set_state(U)
    dt = 0.5 * s.dt_cfl(0.5)
    r = rel(s.residual(), o.residual(U))
    s.rk3_step(dt)
    ri = rel(s.get_state() - U, o.advance(U, dt) - U)
    say(f"  rel L2 residual {r:.3e}, step increment {ri:.3e}")
    assert r < BAR[precision] and ri < BAR[precision]


@pytest.mark.parametrize("n", [1, 4, 5, 9])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("precision", ["fp64", "fp32bulk"])
def test_tri_euler_tiles(p, precision, n):
    corr = {1: "dg", 4: "ga", 5: "hu", 9: "sd"}[n]
    say(f"case: triangle stage, {2 * n * n} elements P{p} {precision} hllc/{corr}")
    m = cases.split_tri_mesh(n, jitter=0.2, seed=n)
    s = TriSolver(m.xy, m.tris, p, periodic=(1.0, 1.0), riemann="hllc", precision=precision, corr=corr)
    o = T.TriTextbook(p, m.xy, m.tris, s.faces, s.normals, riemann="hllc", corr=corr)
    U = _state(m, p, 7 + n)
    s.set_state(U)
    dt = 0.5 * s.dt_cfl(0.5)
    r = rel(s.residual(), o.residual(U))
    s.rk3_step(dt)
    ri = rel(s.get_state() - U, o.advance(U, dt) - U)
    say(f"  rel L2 residual {r:.3e}, step increment {ri:.3e}")
    assert r < BAR[precision] and ri < BAR[precision]


@pytest.mark.parametrize("p,n,viscous,precision", [(1, 110, False, "fp64"), (1, 111, False, "fp64"), (1, 110, True, "fp64"),
                                                   (1, 111, True, "fp64"), (1, 90, True, "fp64"), (1, 91, True, "fp64"),
                                                   (2, 127, True, "fp32bulk"),
                                                   (2, 128, True, "fp32bulk"), (2, 180, False, "fp64"),
                                                   (2, 182, False, "fp64")])
def test_tri_form_by_size(p, n, viscous, precision):
    """Both sides of the element counts (24,576 at P1, 16,384 there with the BR2 terms in FP64, 32,768 and 65,536 at
    P2) from which large meshes take the scalar form of the stage kernels."""
    say(f"case: triangle stage {'viscous' if viscous else 'inviscid'}, {2 * n * n} elements P{p} {precision}")
    m = cases.split_tri_mesh(n, jitter=0.2, seed=n)
    kw = dict(viscous=True, Re=100.0) if viscous else {}
    s = TriSolver(m.xy, m.tris, p, periodic=(1.0, 1.0), riemann="roe", precision=precision, corr="ga", **kw)
    o = T.TriTextbook(p, m.xy, m.tris, s.faces, s.normals, riemann="roe", corr="ga")
    if viscous:
        o.set_viscous(100.0)
    U = _state(m, p, n)
    s.set_state(U)
    r = rel(s.residual(), o.residual(U))
    say(f"  rel L2 {r:.3e}, tiles of {s.info()['elems_per_block']}")
    assert r < BAR[precision]


@pytest.mark.parametrize("p,n,viscous,precision,corr", [
    (1, 111, False, "fp64", "ga"), (1, 111, False, "fp32bulk", "hu"), (2, 182, False, "fp64", "sd"),
    (2, 182, False, "fp32bulk", "ga"), (1, 111, True, "fp64", "hu"), (1, 111, True, "fp32bulk", "ga"),
    (2, 128, True, "fp32bulk", "dg"), (2, 128, True, "fp64", "sd"), (1, 91, True, "fp64", "dg"),
    (2, 148, False, "fp64", "dg"), (2, 156, False, "fp32bulk", "hu"), (2, 158, False, "fp64", "dg")])
def test_tri_large_low_order_steps(p, n, viscous, precision, corr):
    """Two steps of meshes above those counts (and of P2 Euler meshes of 43,808 to 49,928 elements, on both sides of
    the count that the tiles of 64 divide evenly over the CUs): the stage updates, and the traces across tiles that each stage leaves
    for the next and the first step for the second (set_state forms them only once)."""
    say(f"case: triangle steps {'viscous' if viscous else 'inviscid'}, {2 * n * n} elements P{p} {precision} hllc/{corr}")
    m = cases.split_tri_mesh(n, jitter=0.2, seed=n)
    kw = dict(viscous=True, Re=100.0) if viscous else {}
    s = TriSolver(m.xy, m.tris, p, periodic=(1.0, 1.0), riemann="hllc", precision=precision, corr=corr, **kw)
    o = T.TriTextbook(p, m.xy, m.tris, s.faces, s.normals, riemann="hllc", corr=corr)
    if viscous:
        o.set_viscous(100.0)
    U = _state(m, p, n)
    s.set_state(U)
    dt = 0.5 * s.dt_cfl(0.5)
    s.rk3_step(dt)
    s.rk3_step(dt)
    r = rel(s.get_state() - U, o.advance(o.advance(U, dt), dt) - U)
    l2 = abs(s.residual_l2() - np.linalg.norm(s.residual())) / s.residual_l2()
    say(f"  rel L2 of the increment {r:.3e}, tiles of {s.info()['elems_per_block']}")
    assert r < BAR[precision]
    assert l2 < 0.1  # stage 3's residual, a few per cent of a step away from the new state's


@pytest.mark.parametrize("p,n,precision", [(1, 91, "fp32bulk"), (2, 158, "fp64"), (2, 160, "fp32bulk"), (3, 317, "fp64"),
                                           (3, 317, "fp32bulk"), (5, 224, "fp64"), (5, 317, "fp32bulk")])
def test_tri_large_residual(p, n, precision):
    """A residual alone of meshes whose stages take the matrix-core form, in the scalar form with its tiles of 64: the
    traces that steps left for tiles of 32 suffice, and the norm counts the residual's own tiles.  Against the stage
    form's values on the same state and mesh, by the difference a vanishing step makes: dU = dt R to the rounding of
    the state, 1e-16 |U| / (dt |R|)."""
    say(f"case: triangle residual after a step, {2 * n * n} elements P{p} {precision} hllc/ga")
    m = cases.split_tri_mesh(n, jitter=0.2, seed=n)
    s = TriSolver(m.xy, m.tris, p, periodic=(1.0, 1.0), riemann="hllc", precision=precision, corr="ga")
    assert s.info()["elems_per_block"] == 32
    U = _state(m, p, n)
    s.set_state(U)
    dt = 0.5 * s.dt_cfl(0.5)
    s.rk3_step(dt)
    U1 = s.get_state()
    R = s.residual()
    assert abs(s.residual_l2() / np.linalg.norm(R) - 1) < 1e-12
    s.rk3_step(1e-3 * dt)
    d = rel((s.get_state() - U1) / (1e-3 * dt), R)
    rounding = 4e-16 * np.linalg.norm(U1) / (1e-3 * dt * np.linalg.norm(R))
    say(f"  rel L2 {d:.3e}, rounding {rounding:.3e}")
    # the step's own curvature is 1e-3 dt / 2 times the residual's rate of change, of the CFL number's order
    assert d < 5e-4 + rounding + BAR[precision]
    r2 = rel(_residual_of(s, U1), R)
    say(f"  after a trace of every edge {r2:.3e}")
    assert r2 < 1e-13 if precision == "fp64" else r2 < 1e-6


def _residual_of(s, U):
    s.set_state(U)
    return s.residual()


@pytest.mark.parametrize("p,precision", [(1, "fp64"), (1, "fp32bulk"), (2, "fp64")])
def test_tri_large_low_order_boundaries(p, precision):
    """The same with boundary faces (far field, outflow, slip wall and no-slip wall, one type per side)."""
    n = 111 if p == 1 else 182
    say(f"case: triangle steps, open mesh, {2 * n * n} elements P{p} {precision} roe")
    m = cases.split_tri_mesh(n, jitter=0.2, seed=n)
    faces, nrm = tri_faces(m.xy, m.tris)
    side = np.where(np.abs(nrm[:, 0]) > 0.5, np.where(nrm[:, 0] > 0, 6, 4), np.where(nrm[:, 1] > 0, 1, 2))
    bt = np.where(faces[:, 2] < 0, side, 0).astype(np.int32)
    bmap = np.where(bt == 6, 1, 0).astype(np.int32)
    bcd = np.array([[1.1, 0.3, 0.1, 2e3, 0, 0, 0, 0], [2e3, 0, 0, 0, 0, 0, 0, 0]], np.float64)
    s = TriSolver(m.xy, m.tris, p, faces=faces, normals=nrm, bc_type=bt, bc_face_map=bmap, bc_data=bcd, riemann="roe",
                  precision=precision)
    o = T.TriTextbook(p, m.xy, m.tris, faces, nrm, riemann="roe", bc_type=bt, bc_face_map=bmap, bc_data=bcd)
    shp = sp_coords(m.xy, m.tris, p).shape[:2]
    U = cases.perturb(cases.prim_to_cons(np.full(shp, 1.0), np.full(shp, 0.3), np.full(shp, -0.1), np.full(shp, 2e3), 1.4),
                      0.05, 4).reshape(-1)
    s.set_state(U)
    dt = 0.5 * s.dt_cfl(0.5)
    s.rk3_step(dt)
    s.rk3_step(dt)
    r = rel(s.get_state() - U, o.advance(o.advance(U, dt), dt) - U)
    say(f"  rel L2 of the increment {r:.3e}")
    assert r < BAR[precision]


@pytest.mark.parametrize("p,n,precision", [(1, 111, "fp64"), (1, 100, "fp32bulk"), (1, 111, "fp32bulk"), (1, 160, "fp32bulk"),
                                           (2, 100, "fp32bulk"), (2, 128, "fp32bulk")])
def test_tri_large_low_order_viscous_vjp(p, n, precision):
    """The adjoint of meshes around those counts, where the stage's tiles and the adjoint's may differ: two steps
    backwards with dJ/d(dt) (a step's edge cotangents are the next one's input), and the residual's VJP, as
    test_tri_viscous_vjp_tiles has them.  Rounding is independent of g: in a product with a random g over N >= 240,000
    values, divided by the factors' norms, an error of 6e-8 (FP32) over some tens of terms a value enters at
    1e-6 / sqrt(N) = 2e-9, and the difference quotient's 1e-8 at 2e-11."""
    say(f"case: triangle viscous VJP, {2 * n * n} elements P{p} {precision} roe/hu")
    s, o, m = _pair(n, p, "roe", "hu", precision=precision, seed=n)
    U = _state(m, p, 3 + n)
    s.set_state(U)
    dt, eps = 0.25 * s.dt_cfl(0.5), 1e-5
    rng = np.random.default_rng(n)
    g, v = rng.standard_normal(U.size), rng.standard_normal(U.size) * U
    bar = 1e-10 if precision == "fp64" else 1e-8
    scale = np.linalg.norm(g) * np.linalg.norm(v)
    want = float(g @ (o.residual(U + eps * v) - o.residual(U - eps * v))) / (2 * eps)
    scale_r = np.linalg.norm(g) * np.linalg.norm(o.residual(U + eps * v) - o.residual(U - eps * v)) / (2 * eps)
    rr = abs(float(s.residual_vjp(g) @ v) - want) / scale_r
    U1 = o.advance(U, dt)
    s.set_state(U1)
    s.adjoint_set(g)
    dtb = s.rk3_step_vjp(dt)
    s.set_state(U)
    s.rk3_step_vjp(dt, want_dt=False)
    got = float(s.adjoint_get() @ v)

    def two(X):
        return o.advance(o.advance(X, dt), dt)

    want = float(g @ (two(U + eps * v) - two(U - eps * v))) / (2 * eps)
    h = 1e-4 * dt
    want_dt = float(g @ (o.advance(U1, dt + h) - o.advance(U1, dt - h))) / (2 * h)
    scale_dt = np.linalg.norm(g) * np.linalg.norm(o.residual(U1))
    r, rd = abs(got - want) / scale, abs(dtb - want_dt) / scale_dt
    say(f"  residual {rr:.3e}, two steps {r:.3e}, time step {rd:.3e}")
    assert rr < bar and r < bar and rd < bar


@pytest.mark.parametrize("n", [1, 3, 5])
@pytest.mark.parametrize("p,precision", [(1, "fp64"), (2, "fp32bulk"), (3, "fp64"), (4, "fp32bulk"), (5, "fp64"), (5, "fp32bulk")])
def test_tri_viscous_cotangent_unchanged(p, precision, n):
    """A cotangent that no step has taken backwards comes back as it was set, bit for bit, also where the last group
    of elements is not full; and so after the edge cotangents of a step are dropped by a new seed."""
    say(f"case: triangle viscous cotangent, {2 * n * n} elements P{p} {precision}")
    s, _, m = _pair(n, p, "roe", "dg", precision=precision, seed=n)
    U = _state(m, p, n)
    g = np.random.default_rng(n).standard_normal(U.size)
    s.set_state(U)
    s.adjoint_set(g)
    assert np.array_equal(s.adjoint_get(), g)
    s.rk3_step_vjp(0.25 * s.dt_cfl(0.5))
    assert not np.array_equal(s.adjoint_get(), g)
    s.adjoint_set(g)
    assert np.array_equal(s.adjoint_get(), g)


@pytest.mark.parametrize("n", [1, 4, 5])
@pytest.mark.parametrize("p,precision", [(1, "fp64"), (2, "fp64"), (5, "fp64"), (1, "fp32bulk"), (2, "fp32bulk"),
                                         (4, "fp32bulk")])
def test_tri_viscous_vjp_tiles(p, precision, n):
    """One step backwards with dJ/d(dt) at the adjoint's tile edges (32 elements; 64 at P1, 16 at FP64 P5):
    <g, dU1/dU v> and <g, dU1/d(dt)> against central differences of the oracle's step.  The difference
    quotient's own error is eps^2 / 6 times the third derivative plus rounding / eps: 1e-8 at eps = 1e-5;
    FP32-bulk carries its 1e-6 residual error into the product of a random g with the step."""
    corr = {1: "ga", 4: "dg", 5: "hu"}[n]
    say(f"case: triangle viscous step VJP, {2 * n * n} elements P{p} {precision} roe/{corr}")
    s, o, m = _pair(n, p, "roe", corr, precision=precision, seed=n)
    U = _state(m, p, 3 + n)
    s.set_state(U)
    dt, eps = 0.25 * s.dt_cfl(0.5), 1e-5
    rng = np.random.default_rng(n)
    g, v = rng.standard_normal(U.size), rng.standard_normal(U.size) * U
    s.adjoint_set(g)
    dtb = s.rk3_step_vjp(dt)
    got, got_dt = float(s.adjoint_get() @ v), dtb
    want = float(g @ (o.advance(U + eps * v, dt) - o.advance(U - eps * v, dt))) / (2 * eps)
    h = 1e-4 * dt
    want_dt = float(g @ (o.advance(U, dt + h) - o.advance(U, dt - h))) / (2 * h)
    scale, scale_dt = np.linalg.norm(g) * np.linalg.norm(v), np.linalg.norm(g) * np.linalg.norm(o.residual(U))
    r, rd = abs(got - want) / scale, abs(got_dt - want_dt) / scale_dt
    say(f"  state {r:.3e}, time step {rd:.3e}")
    bar = 1e-8 if precision == "fp64" else 1e-5
    assert r < bar and rd < bar
