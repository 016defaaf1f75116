"""Triangle stage kernels at the edges of their element tiles on an MI355X,
against the triangle oracle: a mesh smaller than a wave's group of elements,
exactly one tile (32 elements), a tile and a remainder, several tiles.

Bars: the residual's 1e-12 (FP64) and 1e-5 (FP32-bulk), relative L2.  A step's
increment is a few 1e-3 of the state at these time steps, so the state's
rounding (1e-16 FP64) shows in it at 1e-13 and the bar holds for it too; the
FP32-bulk increment carries the residual's own FP32 error.
"""
import pytest

from tests.test_gpu_parity import rel, say
from tests.test_gpu_tri_viscous import _pair, _state

pytestmark = pytest.mark.gpu

BAR = {"fp64": 1e-12, "fp32bulk": 1e-5}


@pytest.mark.parametrize("n", [1, 4, 5, 9])
@pytest.mark.parametrize("p,precision", [(2, "fp64"), (3, "fp64"), (5, "fp64"), (3, "fp32bulk"), (4, "fp32bulk"), (5, "fp32bulk")])
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
