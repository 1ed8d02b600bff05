"""GPU parity against the oracle, point by point, of the fused elastic / VTI time step
(fwi3d_amd/csrc/fused.hpp, the default form) and of the flux / interior / slab / edge
form. The fused launch updates the planes 6 cells inside the y faces with the stresses
and fluxes of nl_we_op_e / nl_we_op_vti::propagate (src/cpp/we_op.cpp:646-836,
1290-1497) formed on chip, including the x / z closure rows, the traction SATs of the x
and z faces and their absorbing scaling.

The shapes cover each tiling case of an axis (tile widths 16 along x, 32 along z): one
tile, two tiles where the axis is shorter than a tile plus 8 points, and several tiles
with a short middle tile and a last tile shifted to the face; the y chunk of the fused
kernel is forced small so that chunks with remainders occur. Receivers on every grid
node make the traces the whole displacement field at every step (as in
test_gpu_elastic.py). Tolerance: relative L2 <= 1e-4 over all samples and the worst
point of the last sample <= 1e-3 of the field's maximum."""
import numpy as np
import pytest

import fwi3d_amd as F
from oracle import oracle as O

from test_gpu_elastic import CASES, rel, small_shot

pytestmark = pytest.mark.gpu

TRACE_TOL = 1e-4


@pytest.fixture(scope="module")
def eng():
    e = F.Engine(0)
    yield e
    e.close()


def every_point(eng, physics, shape, case, nt=40, fchunk=5):
    model, src, sloc, _, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    ny, nx, nz = shape
    h = d[0]
    iy, ix, iz = np.meshgrid(np.arange(ny), np.arange(nx), np.arange(nz), indexing="ij")
    rloc = np.stack([ix.ravel() * h, iy.ravel() * h, iz.ravel() * h], axis=1).astype(np.float32)
    cfg = CASES[case]
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    eng.tune(fused=True, fchunk=fchunk)
    try:
        got = eng.propagate(physics, model, src, inj, ext, par, d)
    finally:
        eng.tune(fchunk=0)
    return got, (model, src, sloc, rloc, d, dt, cfg)


@pytest.mark.parametrize("physics", ["elastic", "vti"])
@pytest.mark.parametrize("shape,case", [((30, 45, 70), "mixed"), ((24, 20, 36), "free+absorb+taper"),
                                        ((17, 16, 33), "absorb-all"), ((22, 24, 40), "free-all"),
                                        ((13, 40, 31), "mixed")])
def test_fused_every_point_matches_oracle(eng, physics, shape, case):
    nt = 40
    print(f"[fused {physics} every point] shape={shape} case={case} nt={nt}", flush=True)
    got, (model, src, sloc, rloc, d, dt, cfg) = every_point(eng, physics, shape, case, nt=nt)
    oinj, oext = O.Injector(1, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate(physics, model, src, oinj, oext, opar, d, s="f")
    e = rel(got, want)
    last = np.abs(got[:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
    # where the largest difference of the last sample sits (component, y, x, z)
    k = int(np.argmax(np.abs(got[:, :, -1] - want[:, :, -1]).max(axis=0)))
    print(f"  rel L2 vs oracle f32 {e:.2e}, worst point of the last sample {last:.2e} at "
          f"(y,x,z)={np.unravel_index(k, shape)}")
    assert np.isfinite(got).all() and np.abs(want[:, :, -1]).max() > 0
    assert e <= TRACE_TOL
    assert last <= 10 * TRACE_TOL


@pytest.mark.parametrize("physics", ["elastic", "vti"])
@pytest.mark.parametrize("shape,case", [((30, 45, 70), "mixed"), ((17, 16, 33), "absorb-all")])
def test_unfused_every_point_matches_oracle(eng, physics, shape, case):
    """The flux / interior / slab / edge form (fwi3d_tune FWI3D_TUNE_FUSED = 0) at every
    point against the oracle."""
    nt = 40
    print(f"[unfused {physics} every point] shape={shape} case={case} nt={nt}", flush=True)
    model, src, sloc, _, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    ny, nx, nz = shape
    h = d[0]
    iy, ix, iz = np.meshgrid(np.arange(ny), np.arange(nx), np.arange(nz), indexing="ij")
    rloc = np.stack([ix.ravel() * h, iy.ravel() * h, iz.ravel() * h], axis=1).astype(np.float32)
    cfg = CASES[case]
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
    eng.tune(fused=False)
    try:
        got = eng.propagate(physics, model, src, inj, ext, par, d)
    finally:
        eng.tune(fused=True)
    oinj, oext = O.Injector(1, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate(physics, model, src, oinj, oext, opar, d, s="f")
    e = rel(got, want)
    last = np.abs(got[:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
    print(f"  rel L2 vs oracle f32 {e:.2e}, worst point of the last sample {last:.2e}")
    assert np.isfinite(got).all() and e <= TRACE_TOL and last <= 10 * TRACE_TOL


@pytest.mark.parametrize("physics", ["elastic", "vti"])
def test_fused_equals_unfused(eng, physics):
    """The fused step and the flux / interior / slab / edge kernels compute the same
    field to rounding (a larger grid than the every-point cases, default y chunks)."""
    shape, nt = (48, 66, 100), 60
    print(f"[fused vs unfused {physics}] shape={shape} nt={nt}", flush=True)
    model, src, sloc, rloc, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    out = {}
    for fused in (True, False):
        for case in ("mixed", "free+absorb+taper"):
            cfg = CASES[case]
            par = F.make_param(nt, dt, bc=cfg["bc"], taper=cfg["taper"])
            eng.tune(fused=fused)
            try:
                out[fused, case] = eng.propagate(physics, model, src, inj, ext, par, d)
            finally:
                eng.tune(fused=True)
    for case in ("mixed", "free+absorb+taper"):
        e = rel(out[True, case], out[False, case])
        print(f"  {case}: rel L2 fused vs unfused {e:.2e}")
        assert np.isfinite(out[True, case]).all()
        assert e <= 1e-5


@pytest.mark.parametrize("physics", ["elastic", "vti"])
def test_overlap_modes_identical(eng, physics):
    """The fused step's edge tiles (fwi3d_tune FWI3D_TUNE_OVERLAP 3) or y-face launches
    (1, 2) on the second stream, or all on one stream (0), with and without graph replay:
    the launches write disjoint points of the next field, so the traces are bitwise
    equal."""
    shape, nt = (40, 50, 70), 50
    print(f"[overlap modes {physics}] shape={shape} nt={nt}", flush=True)
    model, src, sloc, rloc, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=CASES["mixed"]["bc"], taper=CASES["mixed"]["taper"])
    out = {}
    try:
        for ov in (0, 1, 2, 3):
            for graphs in (True, False):
                eng.tune(overlap=ov, graphs=graphs)
                out[ov, graphs] = eng.propagate(physics, model, src, inj, ext, par, d)
    finally:
        eng.tune(overlap=3, graphs=True)
    ref = out[0, False]
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    for k, v in out.items():
        assert np.array_equal(v, ref), k


@pytest.mark.parametrize("physics", ["elastic", "vti"])
def test_edge_chunks_identical(eng, physics):
    """The y chunk of the fused kernel's side tiles (fwi3d_tune FWI3D_TUNE_ECHUNK; the
    corner tiles take half of it) only changes which workgroup updates a plane: traces
    are bitwise equal for every chunk, including one past the planes' count and the
    autotuner's choice."""
    shape, nt = (40, 50, 70), 40
    print(f"[edge chunks {physics}] shape={shape} nt={nt}", flush=True)
    model, src, sloc, rloc, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    par = F.make_param(nt, dt, bc=CASES["mixed"]["bc"], taper=CASES["mixed"]["taper"])
    out = {}
    try:
        for ec in (0, 1, 5, 8, 13, 100):
            eng.tune(echunk=ec)
            out[ec] = eng.propagate(physics, model, src, inj, ext, par, d)
        eng.tune(echunk=0)
        eng.autotune(physics, shape, steps=2)
        out["auto"] = eng.propagate(physics, model, src, inj, ext, par, d)
    finally:
        eng.tune(echunk=0)
    ref = out[0]
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    for k, v in out.items():
        assert np.array_equal(v, ref), k


@pytest.mark.parametrize("physics", ["elastic", "vti"])
@pytest.mark.parametrize("shape,case", [((12, 12, 12), "mixed"), ((12, 33, 64), "absorb-all"),
                                        ((13, 17, 39), "free-all"), ((20, 56, 104), "mixed"),
                                        ((19, 23, 32), "free+absorb+taper"), ((26, 16, 73), "absorb-all")])
def test_fused_tile_classes_match_oracle(eng, physics, shape, case):
    """The tile classes of the one-launch step at their limits: no plane between the y faces
    (12 planes) or one, axes of one tile, two tiles (33, 39 along z; 17, 23 along x), and
    middle tiles in every row and column of tiles (56 x 104); y chunks of 3 planes with
    remainders. Tolerances as above: relative L2 of rounding over 40 steps."""
    nt = 40
    print(f"[fused classes {physics}] shape={shape} case={case} nt={nt}", flush=True)
    got, (model, src, sloc, rloc, d, dt, cfg) = every_point(eng, physics, shape, case, nt=nt, fchunk=3)
    oinj, oext = O.Injector(1, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    opar = O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"])
    want, _ = O.propagate(physics, model, src, oinj, oext, opar, d, s="f")
    last = np.abs(got[:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
    print(f"  rel L2 vs oracle f32 {rel(got, want):.2e}, worst point of the last sample {last:.2e}")
    assert np.isfinite(got).all() and np.abs(want[:, :, -1]).max() > 0
    assert rel(got, want) <= TRACE_TOL and last <= 10 * TRACE_TOL


def test_narrow_grid_in_the_fixed_workspace(eng):
    """On a narrow grid the fused step's boundary tables exceed the flux buffer: a shot that
    fits the fixed workspace only with the flux buffer still runs there, by the flux form."""
    import torch
    shape, nt = (2280, 12, 64), 6
    d = (0.01, 0.01, 0.01)
    print(f"[narrow workspace] shape={shape}", flush=True)
    dev = torch.device("cuda:0")
    m = torch.stack([torch.full(shape, v, device=dev) for v in (8.0, 6.0, 2.3)]).contiguous()
    src = torch.rand((6, 1, nt), generator=torch.Generator(device=dev).manual_seed(3), device=dev)
    inj = F.Injector(1, np.array([[0.0513, 11.4013, 0.3013]], np.float32), shape, d)
    ext = F.Injector(0, np.array([[0.0613, 11.4113, 0.2913]], np.float32), shape, d)
    par = F.make_param(nt, 0.0008, bc=(1, 2, 2, 2, 2, 2))
    out = []
    for f in (eng.propagate_device, eng.propagate_device_noalloc):
        r = torch.zeros((3, 1, nt), device=dev)
        torch.cuda.synchronize()
        f("elastic", m.data_ptr(), src.data_ptr(), r.data_ptr(), inj, ext, par, shape, d)
        out.append(r.cpu().numpy())
    assert np.abs(out[0]).max() > 0
    assert rel(out[1], out[0]) <= 1e-5  # the two step forms agree to rounding


@pytest.mark.parametrize("physics,shape", [("acoustic", (6700, 12, 64)), ("elastic", (2280, 12, 64)),
                                           ("vti", (1720, 12, 64))])
def test_fixed_workspace_without_boundary_tables(eng, physics, shape):
    """A shot that fits the fixed workspace only without the boundary coefficients takes the
    step of a forward run with a snapshot store: the same kernels in the same order, so the
    same bits."""
    import torch
    nt, d, rng = 24, (0.01, 0.01, 0.01), np.random.default_rng(8)
    ny, nx, nz = shape
    print(f"[workspace limit {physics}] shape={shape}", flush=True)
    dev = torch.device("cuda:0")
    vals = {"acoustic": (8.0, 0.4), "elastic": (8.0, 6.0, 2.3), "vti": (8.0, 6.0, 2.3, 8.2, 0.1, 6.3)}[physics]
    ns, nc = (1, 1) if physics == "acoustic" else (6, 3)
    m = torch.stack([torch.full(shape, v, device=dev) for v in vals]).contiguous()
    src = torch.from_numpy(rng.standard_normal((ns, 1, nt)).astype(np.float32)).to(dev)
    y = ny // 2 * 0.01  # (the y-face slabs are the same kernels in both of the other forms)
    inj = F.Injector(0 if ns == 1 else 1, np.array([[0.0513, y, 0.3013]], np.float32), shape, d)
    ext = F.Injector(0, np.array([[0.0613, y + 0.01, 0.2913], [0.02, y - 0.03, 0.05]], np.float32), shape, d)
    out = []
    for f, sub in ((eng.propagate_device, nt), (eng.propagate_device_noalloc, 0)):
        r = torch.zeros((nc, 2, nt), device=dev)
        torch.cuda.synchronize()
        f(physics, m.data_ptr(), src.data_ptr(), r.data_ptr(), inj, ext,
          F.make_param(nt, 0.0008, sub=sub, bc=(1, 2, 2, 2, 2, 2)), shape, d)
        torch.cuda.synchronize()
        out.append(r.cpu().numpy())
    assert np.isfinite(out[0]).all() and np.abs(out[0]).max() > 0
    assert np.array_equal(out[1], out[0])


@pytest.mark.parametrize("physics", ["elastic", "vti"])
@pytest.mark.parametrize("shape,case", [((12, 12, 12), "mixed"), ((15, 20, 36), "absorb-all"),
                                        ((16, 23, 33), "free-all"), ((30, 45, 104), "free+absorb+taper")])
def test_store_forward_every_point_matches_oracle(eng, physics, shape, case):
    """A forward run that fills a snapshot store takes the step of several launches:
    every point against the oracle, on grids with the whole flux pass (ny < 16) and with the
    y-face one, and bitwise the same on one and on two
    streams and for every store format. Tolerances as above."""
    nt = 40
    print(f"[store {physics}] shape={shape} case={case} nt={nt}", flush=True)
    model, src, sloc, _, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    h = d[0]
    iy, ix, iz = np.meshgrid(*(np.arange(n) for n in shape), indexing="ij")
    rloc = np.stack([ix.ravel() * h, iy.ravel() * h, iz.ravel() * h], axis=1).astype(np.float32)
    cfg = CASES[case]
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    got = []
    try:
        for sp, ov in (("bf16", 0), ("bf16", 1), ("f32", 2), ("f16", 3)):
            eng.tune(overlap=ov)
            par = F.make_param(nt, dt, sub=4, bc=cfg["bc"], taper=cfg["taper"], snap_precision=sp)
            got.append(eng.propagate(physics, model, src, inj, ext, par, d))
    finally:
        eng.tune(overlap=3)
    oinj, oext = O.Injector(1, sloc, shape, d, (0, 0, 0)), O.Injector(0, rloc, shape, d, (0, 0, 0))
    want, _ = O.propagate(physics, model, src, oinj, oext, O.make_par(nt, 0, dt, bc=cfg["bc"], taper=cfg["taper"]),
                          d, s="f")
    last = np.abs(got[0][:, :, -1] - want[:, :, -1]).max() / np.abs(want[:, :, -1]).max()
    print(f"  rel L2 vs oracle f32 {rel(got[0], want):.2e}, worst point of the last sample {last:.2e}")
    assert all(np.array_equal(g, got[0]) for g in got[1:])
    assert np.isfinite(got[0]).all() and np.abs(want[:, :, -1]).max() > 0
    assert rel(got[0], want) <= TRACE_TOL and last <= 10 * TRACE_TOL


def test_wide_face_keeps_32bit_offsets(eng):
    """The boundary coefficients of a VTI face of 3.8 M points pass 4 GiB: such a grid runs the
    step of several launches, with the flux form's results near the far corner of the face
    (rounding of a few steps: 1e-5, as test_fused_equals_unfused)."""
    import torch
    shape, nt, h = (12, 1920, 1984), 12, 0.01
    print(f"[wide face] shape={shape}", flush=True)
    dev = torch.device("cuda:0")
    m = torch.stack([torch.full(shape, v, device=dev) for v in (8.0, 6.0, 2.3, 8.2, 0.1, 6.3)]).contiguous()
    src = torch.rand((6, 1, nt), generator=torch.Generator(device=dev).manual_seed(5), device=dev)
    x, z = (shape[1] - 4) * h, (shape[2] - 4) * h
    inj = F.Injector(1, np.array([[x + 0.003, 0.023, z + 0.004]], np.float32), shape, (h, h, h))
    ext = F.Injector(0, np.array([[x + 0.011, 0.013, z - 0.006], [x - 0.012, 0.041, z]], np.float32), shape, (h, h, h))
    par = F.make_param(nt, 0.0008, bc=(1, 2, 2, 2, 2, 2))
    out = []
    try:
        for fused in (True, False):
            eng.tune(fused=fused)
            r = torch.zeros((3, 2, nt), device=dev)
            torch.cuda.synchronize()
            eng.propagate_device("vti", m.data_ptr(), src.data_ptr(), r.data_ptr(), inj, ext, par, shape, (h, h, h))
            torch.cuda.synchronize()
            out.append(r.cpu().numpy())
    finally:
        eng.tune(fused=True)
    assert np.isfinite(out[0]).all() and np.abs(out[1]).max() > 0
    assert rel(out[0], out[1]) <= 1e-5


def test_two_stream_step_is_launched_directly(eng):
    """The several-launch step without a store (wide faces) is not replayed from a graph: the
    profile counts the y faces' flux pass of every step (a replayed window counts none of its
    kernels)."""
    import torch
    shape, nt, h = (12, 1920, 1984), 35, 0.01  # two windows of 16 steps and a remainder
    print(f"[two streams] shape={shape}", flush=True)
    dev = torch.device("cuda:0")
    m = torch.stack([torch.full(shape, v, device=dev) for v in (8.0, 6.0, 2.3, 8.2, 0.1, 6.3)]).contiguous()
    src = torch.zeros((6, 1, nt), device=dev)
    inj = F.Injector(1, np.array([[1.003, 0.053, 1.004]], np.float32), shape, (h, h, h))
    ext = F.Injector(0, np.zeros((0, 3), np.float32), shape, (h, h, h))
    torch.cuda.synchronize()
    eng.profile(True)
    try:
        eng.propagate_device("vti", m.data_ptr(), src.data_ptr(), 0, inj, ext, F.make_param(nt, 0.0008), shape, (h, h, h))
        n = eng.profile_read(1)[1]
    finally:
        eng.profile(False)
    assert n == nt - 1


@pytest.mark.parametrize("physics", ["elastic", "vti"])
def test_profile_classes_of_the_two_step_forms(eng, physics):
    """Class 0 is the one-launch step; a forward run with a store counts its fused tiles as class
    5 and its y faces as classes 1 and 3."""
    shape, nt = (30, 34, 38), 21
    model, src, sloc, rloc, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
    inj, ext = F.Injector(1, sloc, shape, d), F.Injector(0, rloc, shape, d)
    got = {}
    try:
        for sub in (0, 4):
            eng.tune(graphs=False)
            eng.profile(True)
            eng.propagate(physics, model, src, inj, ext, F.make_param(nt, dt, sub=sub), d)
            got[sub] = [eng.profile_read(k)[1] for k in (0, 1, 2, 3, 5)]
    finally:
        eng.profile(False)
        eng.tune(graphs=True)
    assert got[0] == [nt - 1, 0, 0, 0, 0]
    assert got[4] == [0, nt - 1, 0, nt - 1, nt - 1]


@pytest.mark.parametrize("physics", ["acoustic", "elastic", "vti"])
def test_traces_with_and_without_a_store(eng, physics):
    """A forward run that fills a store takes another step form than one without: the traces agree
    to rounding (1e-5, as the step forms above), do not depend on the interval, and are the same
    bits where both run the flux / interior form."""
    shape, nt = (40, 50, 70), 100
    if physics == "acoustic":
        from fwi3d_amd import workloads as W
        _, _, sloc, rloc, d, dt = small_shot("elastic", 1, shape=shape, nt=nt)
        vp = (1.8 + 0.6 * W.smooth_random(shape, 4, 3)).astype(np.float32)
        model, src, kind = W.acoustic_convert(vp, W.gardner(vp)), W.ricker(25, nt, dt)[None, None, :].astype(np.float32), 0
    else:
        model, src, sloc, rloc, d, dt = small_shot(physics, 1, shape=shape, nt=nt)
        kind = 1
    inj, ext = F.Injector(kind, sloc, shape, d), F.Injector(0, rloc, shape, d)
    cfg = CASES["free+absorb+taper"]
    r = {}
    try:
        for fused in (True, False):
            eng.tune(fused=fused)
            for sub in (0, 1, 7):
                r[fused, sub] = eng.propagate(physics, model, src, inj, ext,
                                              F.make_param(nt, dt, sub=sub, bc=cfg["bc"], taper=cfg["taper"]), d)
    finally:
        eng.tune(fused=True)
    e = rel(r[True, 0], r[True, 7])
    print(f"  {physics}: rel L2 without against with a store {e:.1e}")
    assert np.isfinite(r[True, 0]).all() and np.abs(r[True, 0]).max() > 0
    assert e <= 1e-5
    assert np.array_equal(r[True, 1], r[True, 7])
    assert np.array_equal(r[False, 0], r[False, 1]) and np.array_equal(r[False, 0], r[False, 7])
