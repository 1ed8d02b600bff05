"""The imaging condition (fwi3d_amd/csrc/imaging.hpp) at the edges of its tiles (16 x points,
32 z points, chunks of planes along y) against the oracle: axes of one tile, of a tile plus
less than 8 points, of several tiles with a short middle one, the closure rows of every face.

Tolerances: relative L2 of each gradient <= 1e-3, as the other gradient tests (traces agree to
1e-4, a gradient is a product of two fields); the worst point <= 1e-2 of the largest value
(the same ratio of point to L2 as the traces' tests have)."""
import numpy as np
import pytest

import fwi3d_amd as F
from oracle import oracle as O

import test_gpu_acoustic as TA
import test_gpu_elastic as TE

pytestmark = pytest.mark.gpu
GRAD_TOL = 1e-3


@pytest.fixture(scope="module")
def eng():
    e = F.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("physics", ["acoustic", "elastic", "vti"])
@pytest.mark.parametrize("shape", [(12, 12, 12), (13, 16, 32), (17, 17, 33), (21, 23, 39), (24, 24, 40), (14, 41, 72)])
def test_gradient_at_tile_edges(eng, physics, shape):
    nt, sub, dt = 121, 4, 0.0008
    print(f"[imaging {physics}] shape={shape}", flush=True)
    if physics == "acoustic":
        model, src, sloc, rloc, d = TA.small_shot(shape=shape, nt=nt, dt=dt)
        ng, kind = 2, 0
    else:
        model, src, sloc, rloc, d, _ = TE.small_shot(physics, 1, shape=shape, nt=nt, dt=dt)
        ng, kind = 3, 1
    bc, taper = (1, 2, 2, 2, 2, 2), (0, 3, 3, 3, 3, 3)
    inj, ext = F.Injector(kind, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, sub=sub, bc=bc, taper=taper)
    rcv = eng.propagate(physics, model, src, inj, ext, par, d)
    res = np.ascontiguousarray(rcv[:, :, ::-1] * 0.5)
    grad = np.zeros((ng,) + shape, np.float32)
    eng.propagate(physics, model, res, ext, None, par, d, adj=True, grad=grad)
    oinj, oext = O.Injector(kind, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, sub, dt, bc=bc, taper=taper)
    _, snaps = O.propagate(physics, model, src, oinj, oext, opar, d, s="f")
    want = np.zeros((ng,) + shape, np.float32)
    O.propagate(physics, model, res, oext, oinj, opar, d, adj=True, grad=want, snaps=snaps, s="f")
    for k in range(ng):
        e, worst = TE.rel(grad[k], want[k]), np.abs(grad[k] - want[k]).max() / np.abs(want[k]).max()
        print(f"  grad[{k}] rel L2 {e:.2e}, worst point {worst:.2e}")
        assert np.isfinite(grad[k]).all() and e <= GRAD_TOL and worst <= 10 * GRAD_TOL
