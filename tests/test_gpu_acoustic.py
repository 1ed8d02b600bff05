"""GPU parity of the acoustic path (nl_we_op_a::propagate, src/cpp/we_op.cpp:1607-1827)
through the C ABI, against the oracle on the same inputs.

Tolerances (north_star): traces relative L2 <= 1e-4 against the single-precision
oracle; gradients relative L2 <= 1e-3."""
import os

import numpy as np
import pytest

import fwi3d_amd as F
from fwi3d_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
TRACE_TOL = 1e-4
GRAD_TOL = 1e-3


def rel(a, b):
    return float(np.linalg.norm((np.asarray(a, np.float64) - b).ravel()) / np.linalg.norm(np.asarray(b, np.float64).ravel()))


@pytest.fixture(scope="module")
def eng():
    e = F.Engine(0)
    yield e
    e.close()


def small_shot(shape=(36, 40, 44), nt=300, dt=0.001, h=0.01, seed=3):
    """Smooth random acoustic model, a source off-centre and receivers spread over the
    box including points next to every face."""
    ny, nx, nz = shape
    rng = np.random.default_rng(seed)
    vp = (1.6 + 0.8 * W.smooth_random(shape, 4, seed)).astype(np.float32)
    rho = W.gardner(vp) * (1 + 0.1 * W.smooth_random(shape, 3, seed + 1)).astype(np.float32)
    model = W.acoustic_convert(vp, rho)
    src = W.ricker(25.0, nt, dt)[None, None, :]
    sloc = np.array([[0.47 * (nx - 1) * h, 0.52 * (ny - 1) * h, 0.37 * (nz - 1) * h]], np.float32)
    L = np.array([(nx - 1) * h, (ny - 1) * h, (nz - 1) * h])
    pts = [rng.uniform(0, 1, 3) * L for _ in range(40)]
    for ax in range(3):
        for end in (0.0, 1.0):
            p = rng.uniform(0.2, 0.8, 3) * L
            p[ax] = end * L[ax]
            pts.append(p)
    rloc = np.array(pts, np.float32)
    return model, src, sloc, rloc, (h, h, h)


CASES = {
    "free+absorb+taper": dict(bc=(1, 2, 2, 2, 2, 2), taper=(0, 8, 8, 8, 8, 8)),
    "absorb-all+taper": dict(bc=(2, 2, 2, 2, 2, 2), taper=(5, 5, 5, 5, 5, 5)),
    "free-all": dict(bc=(1, 1, 1, 1, 1, 1), taper=(0,) * 6),
    "mixed": dict(bc=(3, 2, 1, 3, 0, 2), taper=(0, 4, 0, 6, 3, 0)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_acoustic_forward_matches_oracle(eng, case):
    model, src, sloc, rloc, d = small_shot()
    cfg = CASES[case]
    nt, dt = src.shape[-1], 0.001
    shape = model.shape[-3:]
    print(f"[acoustic fwd] case={case} shape={shape} nt={nt}", flush=True)
    inj, ext = F.Injector(0, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    got = eng.propagate("acoustic", model, src, inj, ext, par, d)

    oinj, oext = O.Injector(0, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate("acoustic", model, src, oinj, oext, opar, d, s="f")
    want64, _ = O.propagate("acoustic", model.astype(np.float64), src.astype(np.float64), oinj.as_double(),
                            oext.as_double(), opar, d, s="d")
    e32, e64, o64 = rel(got, want), rel(got, want64), rel(want, want64)
    print(f"  rel L2 vs oracle f32 {e32:.2e}, vs f64 {e64:.2e} (oracle f32 vs f64 {o64:.2e})")
    assert np.isfinite(got).all() and np.abs(want).max() > 0
    assert e32 <= TRACE_TOL
    assert e64 <= max(TRACE_TOL, 3 * o64)


def test_acoustic_config_a_full_size(eng):
    """Config A at full size (100^3, nt=1000) against the committed oracle traces."""
    s = W.config_a()
    print(f"[acoustic config A] shape={s.shape} nt={s.nt}", flush=True)
    inj, ext = F.Injector(0, s.src_loc, s.shape, s.d), F.Injector(0, s.rcv_loc, s.shape, s.d)
    par = F.make_param(s.nt, s.dt, bc=s.bc, taper=s.taper, taper_strength=s.taper_strength)
    got = eng.propagate("acoustic", s.model, s.src, inj, ext, par, s.d)
    want = np.load(os.path.join(GOLDEN, "config_a_traces_f32.npy"))
    want64 = np.load(os.path.join(GOLDEN, "config_a_traces_f64.npy"))
    e32, e64, o64 = rel(got, want), rel(got, want64), rel(want, want64)
    print(f"  rel L2 vs oracle f32 {e32:.2e}, vs f64 {e64:.2e} (oracle f32 vs f64 {o64:.2e})")
    assert e32 <= TRACE_TOL
    assert e64 <= max(TRACE_TOL, 3 * o64)


@pytest.mark.parametrize("sub", [3, 4])
def test_acoustic_gradient_matches_oracle(eng, sub):
    """Forward with snapshots every `sub` steps, then the adjoint with a residual
    injected at the receivers; imaging condition (gK, g(1/rho)) vs the oracle.
    nt=201 with sub=4 hits the (nt-1)%sub==0 'last sample' branch, sub=3 the
    zero-slot branch."""
    model, src, sloc, rloc, d = small_shot(nt=201)
    nt, dt = 201, 0.001
    shape = model.shape[-3:]
    cfg = CASES["free+absorb+taper"]
    print(f"[acoustic grad] sub={sub} shape={shape} nt={nt}", flush=True)
    inj, ext = F.Injector(0, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, sub=sub, bc=cfg["bc"], taper=cfg["taper"])
    rcv = eng.propagate("acoustic", model, src, inj, ext, par, d)
    res = np.ascontiguousarray(rcv[:, :, ::-1] * 0.7)  # any residual-shaped input
    grad = np.zeros((2,) + shape, np.float32)
    eng.propagate("acoustic", model, res, ext, None, par, d, adj=True, grad=grad)

    oinj, oext = O.Injector(0, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, sub, dt, bc=cfg["bc"], taper=cfg["taper"])
    orcv, snaps = O.propagate("acoustic", model, src, oinj, oext, opar, d, s="f")
    assert rel(rcv, orcv) <= TRACE_TOL
    ograd = np.zeros((2,) + shape, np.float32)
    O.propagate("acoustic", model, res, oext, oinj, opar, d, adj=True, grad=ograd, snaps=snaps, s="f")
    for k in range(2):
        e = rel(grad[k], ograd[k])
        print(f"  grad[{k}] rel L2 {e:.2e}")
        assert e <= GRAD_TOL


@pytest.mark.parametrize("shape,case", [((19, 17, 45), "mixed"), ((19, 26, 70), "free+absorb+taper"),
                                        # an axis of exactly 12 points: no interior tiles, so the
                                        # interior/shell/receiver single launch gives way to the shell kernel
                                        ((40, 12, 30), "mixed"), ((40, 12, 12), "mixed")])
def test_acoustic_every_point_matches_oracle(eng, shape, case):
    """Receivers on every grid node (quadratic extraction weights reduce to the node
    value): the whole pressure field at every step against the oracle, through the
    single-launch step (interior tiles, shell and receivers in one launch) on odd shapes."""
    nt = 60
    model, src, sloc, _, d = small_shot(shape=shape, nt=nt)
    ny, nx, nz = shape
    h = d[0]
    iy, ix, iz = np.meshgrid(np.arange(ny), np.arange(nx), np.arange(nz), indexing="ij")
    rloc = np.stack([ix.ravel() * h, iy.ravel() * h, iz.ravel() * h], axis=1).astype(np.float32)
    cfg = CASES[case]
    dt = 0.001
    print(f"[acoustic every point] shape={shape} case={case} nt={nt}", flush=True)
    inj, ext = F.Injector(0, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    got = eng.propagate("acoustic", model, src, inj, ext, par, d)
    oinj, oext = O.Injector(0, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate("acoustic", model, src, oinj, oext, opar, d, s="f")
    e = rel(got, want)
    last = np.abs(got[:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
    print(f"  rel L2 vs oracle f32 {e:.2e}, worst point of the last sample {last:.2e}")
    assert np.isfinite(got).all() and np.abs(want[:, :, -1]).max() > 0
    assert e <= TRACE_TOL
    assert last <= 10 * TRACE_TOL


@pytest.mark.parametrize("shape,case", [((12, 12, 12), "mixed"), ((13, 16, 32), "absorb-all+taper"), ((17, 17, 33), "free-all"),
                                        ((25, 23, 39), "mixed"), ((24, 24, 40), "free+absorb+taper"), ((26, 41, 72), "mixed")])
@pytest.mark.parametrize("ychunk", [0, 5])
def test_fused_step_every_point_matches_oracle(eng, shape, case, ychunk):
    """The one-launch step at the edges of its tiles (16 x, 32 z points, chunks of planes): the
    whole field at every step, with sources whose stencils overlap (one pair inside a tile, one
    across a tile's edge, one at a face); and the same with the interior / shell kernels. The
    tolerance is that of the traces; the worst point of the last sample within 10 times it."""
    nt, dt = 60, 0.001
    print(f"[acoustic fused] shape={shape} case={case} ychunk={ychunk}", flush=True)
    model, _, _, _, d = small_shot(shape=shape, nt=nt)
    ny, nx, nz = shape
    h = d[0]
    pts = [(0.5 * (nx - 1), 0.5 * (ny - 1), 0.4 * (nz - 1)), (min(nx - 1, 15.6), 0.3 * (ny - 1), min(nz - 1, 31.4)), (0.3, 0.2, 0.1)]
    sloc = np.array([[x * h, y * h, z * h] for x, y, z in pts for _ in range(2)], np.float32)
    sloc[1::2] += np.float32(0.6 * h) * np.sign((np.array([nx, ny, nz]) - 1) * h / 2 - sloc[1::2])
    sloc = np.clip(sloc, 0, (np.array([nx, ny, nz], np.float32) - 1) * np.float32(h))
    rng = np.random.default_rng(2)
    src = (W.ricker(25.0, nt, dt)[None, None, :] * rng.uniform(0.5, 1.5, (1, len(sloc), 1))).astype(np.float32)
    iy, ix, iz = np.meshgrid(*(np.arange(n) for n in shape), indexing="ij")
    rloc = np.stack([ix.ravel() * h, iy.ravel() * h, iz.ravel() * h], axis=1).astype(np.float32)
    cfg = CASES[case]
    inj, ext = F.Injector(0, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate("acoustic", model, src, O.Injector(0, sloc, shape, d, (0, 0, 0)),
                          O.Injector(0, rloc, shape, d, (0, 0, 0)), O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"]),
                          d, s="f")
    assert np.abs(want[:, :, -1]).max() > 0
    for fused in (True, False):
        eng.tune(fused=fused, ychunk=ychunk)
        try:
            got = eng.propagate("acoustic", model, src, inj, ext, par, d)
        finally:
            eng.tune(fused=True, ychunk=0)
        last = np.abs(got[:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
        print(f"  fused={fused}: rel L2 vs oracle {rel(got, want):.2e}, worst point of the last sample {last:.2e}")
        assert np.isfinite(got).all() and rel(got, want) <= TRACE_TOL and last <= 10 * TRACE_TOL


@pytest.mark.parametrize("npts", [1, 2, 3, 5, 38])
def test_overlapping_sources_alone_and_in_a_batch(eng, npts):
    """Sources within two cells of each other, up to some hundred contributions to a point: traces
    against the oracle, and a batched shot with the same bits."""
    import torch
    nt, dt = 80, 0.001
    model, _, _, rloc, d = small_shot(nt=nt)
    shape = model.shape[-3:]
    rng = np.random.default_rng(npts)
    sloc = (np.array([0.19, 0.17, 0.16]) + rng.uniform(0, 2 * d[0], (npts, 3))).astype(np.float32)
    src = (W.ricker(25.0, nt, dt)[None, None, :] * rng.uniform(0.5, 1.5, (1, npts, 1))).astype(np.float32)
    cfg = CASES["free+absorb+taper"]
    inj, ext = F.Injector(0, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    got = eng.propagate("acoustic", model, src, inj, ext, par, d)
    want, _ = O.propagate("acoustic", model, src, O.Injector(0, sloc, shape, d, (0, 0, 0)),
                          O.Injector(0, rloc, shape, d, (0, 0, 0)), O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"]),
                          d, s="f")
    print(f"  {npts} sources: rel L2 vs oracle {rel(got, want):.2e}")
    assert np.abs(want).max() > 0 and rel(got, want) <= TRACE_TOL
    m, s = torch.from_numpy(np.ascontiguousarray(model)).to("cuda:0"), torch.from_numpy(src).to("cuda:0")
    r = torch.zeros((1, ext.npts, nt), device="cuda:0")
    torch.cuda.synchronize()
    b = F.Batch(eng)
    b.add("acoustic", m.data_ptr(), s.data_ptr(), r.data_ptr(), inj, ext, par, shape, d)
    b.run()
    b.close()
    assert np.array_equal(r.cpu().numpy(), got)


def test_dense_receivers_do_not_slow_the_adjoint_step(eng):
    """Four receivers per grid point of a plane, injected by an adjoint run (some hundred
    contributions per point): the one-launch step takes no longer than the interior / shell
    step with an injection launch."""
    import torch
    n, nr, nt, h = 100, 200, 66, 0.01
    shape, d = (n, n, n), (h, h, h)
    dev = torch.device("cuda:0")
    m = torch.stack([torch.full(shape, v, device=dev) for v in (8.0, 0.4)]).contiguous()
    a = np.linspace(0.05, 0.95, nr) * (n - 1) * h
    g1, g2 = np.meshgrid(a, a)
    inj = F.Injector(0, np.stack([g1.ravel(), 0 * g1.ravel() + 0.5 * (n - 1) * h, g2.ravel()], 1).astype(np.float32), shape, d)
    src = torch.rand((1, nr * nr, nt), device=dev)
    torch.cuda.synchronize()
    us = {}
    try:
        for fused in (True, False):
            eng.tune(fused=fused)
            best = 1e30
            for _ in range(3):
                eng.profile(True, steps_only=True)
                eng.propagate_device("acoustic", m.data_ptr(), src.data_ptr(), 0, inj, None,
                                     F.make_param(nt, 0.0005, bc=(1, 2, 2, 2, 2, 2)), shape, d, adj=True)
                ms, k = eng.profile_read(4)  # (replayed windows: the injection included)
                best = min(best, 1e3 * ms / k)
            us[fused] = best
    finally:
        eng.profile(False)
        eng.tune(fused=True)
    print(f"  us per step: one launch {us[True]:.1f}, interior / shell and injection {us[False]:.1f}")
    assert us[True] <= 1.1 * us[False]
