"""Batched forward modelling (fwi3d_batch_*): shots of the three physics on uneven grids,
with different nt and joining the batch at different steps, advance together one
launch per kernel class and step. Each shot's traces in the mix equal, bit for bit, its
traces when it runs alone in a batch, and agree with the single-shot path
(fwi3d_propagate_device, itself held to the oracle) to 1e-6 relative L2."""
import numpy as np
import pytest

import fwi3d_amd as F
from fwi3d_amd import workloads as W

pytestmark = pytest.mark.gpu

H = 0.01
DT = 0.0008


def make_shot(physics, shape, nt, seed):
    rng = np.random.default_rng(seed)
    ny, nx, nz = shape
    vp = (2.0 + 1.3 * W.smooth_random(shape, 4, seed)).astype(np.float32)
    rho = W.gardner(vp)
    if physics == "acoustic":
        model, ns, kind = W.acoustic_convert(vp, rho), 1, 0
    elif physics == "elastic":
        model, ns, kind = W.elastic_convert(vp, vp / 1.8, rho), 6, 1
    else:
        eps = (0.2 * W.smooth_random(shape, 3, seed + 2)).astype(np.float32)
        dlt = (0.1 * W.smooth_random(shape, 3, seed + 3)).astype(np.float32)
        model, ns, kind = W.vti_convert(vp, vp / 2, rho, dlt, eps, 0 * eps), 6, 1
    w = W.ricker(25.0, nt, DT)
    src = (np.stack([w * (1.0 + 0.1 * k) for k in range(ns)])[:, None, :]).astype(np.float32)
    L = np.array([(nx - 1) * H, (ny - 1) * H, (nz - 1) * H])
    sloc = [list(rng.uniform(0.3, 0.7, 3) * L)]
    rloc = [list(rng.uniform(0.05, 0.95, 3) * L) for _ in range(20)]
    inj = F.Injector(kind, sloc, shape, (H, H, H))
    ext = F.Injector(0, rloc, shape, (H, H, H))
    bc = (1, 2, 2, 2, 2, 2) if seed % 2 else (2, 1, 0, 2, 1, 2)
    taper = (0, 5, 5, 5, 5, 5) if seed % 2 else (3, 0, 4, 0, 0, 5)
    par = F.make_param(nt, DT, sub=0, bc=bc, taper=taper)
    return dict(physics=physics, shape=shape, model=model, src=src, inj=inj, ext=ext, par=par)


SHOTS = [
    ("acoustic", (40, 44, 48), 120, 1),
    ("elastic", (30, 34, 38), 100, 2),
    ("vti", (28, 26, 40), 90, 3),
    ("acoustic", (36, 30, 70), 75, 4),
    ("elastic", (20, 27, 66), 110, 5),
    ("vti", (20, 27, 66), 80, 6),
    ("elastic", (40, 12, 30), 70, 7),   # an axis of 12 points: no interior tiles
    ("acoustic", (40, 12, 12), 60, 8),
]


def single(eng, s, dev):
    import torch
    m = torch.from_numpy(s["model"]).to(dev)
    src = torch.from_numpy(s["src"]).to(dev)
    rcv = torch.zeros((F.n_comp(F.PHYSICS[s["physics"]]), s["ext"].npts, s["par"].nt), dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    eng.propagate_device(s["physics"], m.data_ptr(), src.data_ptr(), rcv.data_ptr(), s["inj"], s["ext"], s["par"],
                         s["shape"], (H, H, H))
    torch.cuda.synchronize()
    return rcv.cpu().numpy()


def run_batch(eng, shots, idx, join_late, dev, tune_window=0):
    """Run shots[idx] in one batch; join_late maps a shot index to the global step at
    which it joins (others join at step 0); tune_window > 0 arms the online tile tuner
    (the tiling changes during the run). Returns {index: traces}."""
    import torch
    b = F.Batch(eng)
    if tune_window:
        b.autotune(tune_window)
    keep, ids, out = [], [], {}

    def admit(i):
        s = shots[i]
        m = torch.from_numpy(s["model"]).to(dev)
        src = torch.from_numpy(s["src"]).to(dev)
        rcv = torch.zeros((F.n_comp(F.PHYSICS[s["physics"]]), s["ext"].npts, s["par"].nt), dtype=torch.float32,
                          device=dev)
        torch.cuda.synchronize()
        keep.extend([m, src])
        out[i] = rcv
        ids.append(b.add(s["physics"], m.data_ptr(), src.data_ptr(), rcv.data_ptr(), s["inj"], s["ext"], s["par"],
                         s["shape"], (H, H, H)))

    late = {i: t for i, t in join_late.items() if i in idx}
    for i in idx:
        if i not in late:
            admit(i)
    step = 0
    for i, t in sorted(late.items(), key=lambda x: x[1]):
        b.step(t - step)
        step = t
        admit(i)
    n, resident, it = b.status()
    assert n == len(idx) and resident > 0 and it == step
    b.run()
    assert all(b.query(sid) == 1 for sid in ids)
    assert b.status()[0] == 0 and b.status()[1] == 0
    if tune_window:
        yc, ms = b.tiles()
        print(f"  online tuning: y chunk {yc}, ms/step {['%.3f' % t for t in ms]}", flush=True)
        assert yc in (4, 8, 16, 32) and all(t > 0 for t in ms)
    b.close()
    return {i: r.cpu().numpy() for i, r in out.items()}


def test_batch_mix_equals_alone_and_single_path():
    import torch
    dev = torch.device("cuda:0")
    shots = [make_shot(*a) for a in SHOTS]
    eng = F.Engine(0)
    try:
        join_late = {4: 25, 5: 40}  # shot index -> global step at which it joins
        # the mixed run also re-tiles itself during its first 12 steps (online tuning)
        mixed = run_batch(eng, shots, list(range(len(shots))), join_late, dev, tune_window=3)
        for i in range(len(shots)):
            alone = run_batch(eng, shots, [i], {}, dev)[i]
            want = single(eng, shots[i], dev)
            e = float(np.linalg.norm(mixed[i] - want) / np.linalg.norm(want))
            print(f"  shot {i} {SHOTS[i][0]} {SHOTS[i][1]} nt={SHOTS[i][2]}: mix vs alone max|d| "
                  f"{np.abs(mixed[i] - alone).max():.1e}, batch vs single-shot path rel L2 {e:.2e}", flush=True)
            assert np.abs(want).max() > 0
            # same kernels, same inputs: the other shots in the batch change nothing
            assert np.array_equal(mixed[i], alone), i
            # separately compiled kernels of the single-shot path may contract multiply-adds
            # differently; both are held to the oracle at 1e-4 elsewhere
            assert e <= 1e-6, i
    finally:
        eng.close()


GRAD_SHOTS = [  # physics, shape, nt, seed, sub, snapshot precision
    ("elastic", (30, 34, 38), 100, 12, 4, "f32"),   # (nt-1) % sub != 0: a zero slot, as in the reference
    ("acoustic", (40, 44, 48), 91, 11, 3, "f32"),
    ("vti", (28, 26, 40), 81, 13, 4, "bf16"),
]


def test_batch_gradient_shots_equal_single_path():
    """Forward shots with a snapshot store and their adjoint shots, mixed with a plain
    forward shot, give the traces and FP64 gradients of fwi3d_propagate_device
    (forward with sub > 0, then adjoint on the same context) bit for bit."""
    import torch
    dev = torch.device("cuda:0")
    eng = F.Engine(0)
    try:
        cases = []
        for ph, shape, nt, seed, sub, fmt in GRAD_SHOTS:
            s = make_shot(ph, shape, nt, seed)
            s["par"] = F.make_param(nt, DT, sub=sub, bc=s["par"].bc, taper=s["par"].taper, snap_precision=fmt)
            rng = np.random.default_rng(seed + 100)
            nc = F.n_comp(F.PHYSICS[ph])
            asrc = (rng.standard_normal((nc, s["ext"].npts, nt)) * np.hanning(nt)).astype(np.float32)
            m = torch.from_numpy(s["model"]).to(dev)
            src = torch.from_numpy(s["src"]).to(dev)
            a = torch.from_numpy(asrc).to(dev)
            ng = F.n_grad(F.PHYSICS[ph])
            rcv1 = torch.zeros((nc, s["ext"].npts, nt), dtype=torch.float32, device=dev)
            g1 = torch.zeros((ng,) + shape, dtype=torch.float64, device=dev)
            torch.cuda.synchronize()
            print(f"  single path: {ph} {shape} nt={nt} sub={sub} {fmt}", flush=True)
            eng.propagate_device(ph, m.data_ptr(), src.data_ptr(), rcv1.data_ptr(), s["inj"], s["ext"], s["par"], shape,
                                 (H, H, H))
            eng.propagate_device(ph, m.data_ptr(), a.data_ptr(), 0, s["ext"], s["inj"], s["par"], shape, (H, H, H),
                                 adj=True, grad64_ptr=g1.data_ptr())
            torch.cuda.synchronize()
            cases.append(dict(s=s, m=m, src=src, a=a, rcv1=rcv1, g1=g1, rcv2=torch.zeros_like(rcv1),
                              g2=torch.zeros_like(g1)))
        plain = make_shot("acoustic", (36, 30, 70), 75, 4)
        pm = torch.from_numpy(plain["model"]).to(dev)
        psrc = torch.from_numpy(plain["src"]).to(dev)
        prcv = torch.zeros((1, plain["ext"].npts, 75), dtype=torch.float32, device=dev)
        torch.cuda.synchronize()
        print("  batch: 3 gradient shots + 1 plain shot", flush=True)
        b = F.Batch(eng)
        fwd = {}
        for k, c in enumerate(cases):
            s = c["s"]
            sid = b.add(s["physics"], c["m"].data_ptr(), c["src"].data_ptr(), c["rcv2"].data_ptr(), s["inj"], s["ext"],
                        s["par"], s["shape"], (H, H, H))
            fwd[sid] = k
            fp = F.Batch.snap_footprint(s["physics"], s["shape"], s["par"].nt, s["par"].sub, s["par"].snap_precision)
            assert fp > 0
        b.add("acoustic", pm.data_ptr(), psrc.data_ptr(), prcv.data_ptr(), plain["inj"], plain["ext"], plain["par"],
              plain["shape"], (H, H, H))
        # an adjoint shot may not start before its forward shot has left
        k0 = next(iter(fwd))
        c0 = cases[fwd[k0]]
        with pytest.raises(RuntimeError, match="has not left"):
            b.add_adjoint(k0, c0["s"]["physics"], c0["m"].data_ptr(), c0["a"].data_ptr(), c0["s"]["ext"],
                          c0["g2"].data_ptr(), c0["s"]["par"], c0["s"]["shape"], (H, H, H))
        adj_started, guard = 0, 0
        while b.step(1) > 0 or adj_started < len(cases):
            guard += 1
            assert guard < 1000, "batch did not drain"
            for sid in b.retired():
                if sid in fwd:
                    c = cases[fwd[sid]]
                    s = c["s"]
                    b.add_adjoint(sid, s["physics"], c["m"].data_ptr(), c["a"].data_ptr(), s["ext"], c["g2"].data_ptr(),
                                  s["par"], s["shape"], (H, H, H))
                    adj_started += 1
        b.wait()
        assert b.status()[0] == 0 and b.status()[1] == 0  # shots and snapshot stores all freed
        b.close()
        for c in cases:
            s = c["s"]
            r1, r2 = c["rcv1"].cpu().numpy(), c["rcv2"].cpu().numpy()
            g1, g2 = c["g1"].cpu().numpy(), c["g2"].cpu().numpy()
            print(f"  {s['physics']} {s['shape']}: traces max|d| {np.abs(r1 - r2).max():.1e}, gradient max|d| "
                  f"{np.abs(g1 - g2).max():.1e} (|g| max {np.abs(g1).max():.2e})", flush=True)
            assert np.abs(g1).max() > 0
            assert np.array_equal(r1, r2)
            assert np.array_equal(g1, g2)
    finally:
        eng.close()


def test_batch_snapshot_store_errors_and_footprint():
    import torch
    dev = torch.device("cuda:0")
    s = make_shot("elastic", (24, 24, 24), 40, 7)
    fp = F.Batch.footprint("elastic", s["shape"], s["inj"], s["ext"])
    ny, nx, nz = s["shape"]
    assert fp >= 3 * 3 * ny * nx * 64 * 4  # three 3-component wavefields at a 64-float z pitch
    sfp = F.Batch.snap_footprint("elastic", s["shape"], 40, 4, "f32")
    assert sfp >= 11 * 3 * ny * nx * 64 * 4  # 1 + nt/sub slots of 3 components
    assert F.Batch.snap_footprint("elastic", s["shape"], 40, 4, "bf16") < sfp
    eng = F.Engine(0)
    try:
        b = F.Batch(eng)
        m = torch.from_numpy(s["model"]).to(dev)
        src = torch.from_numpy(s["src"]).to(dev)
        rcv = torch.zeros((3, s["ext"].npts, 40), dtype=torch.float32, device=dev)
        g = torch.zeros((3, ny, nx, nz), dtype=torch.float64, device=dev)
        par = F.make_param(40, DT, sub=4)
        sid = b.add("elastic", m.data_ptr(), src.data_ptr(), rcv.data_ptr(), s["inj"], s["ext"], par, s["shape"],
                    (H, H, H))
        assert b.status()[1] >= fp + sfp
        with pytest.raises(RuntimeError, match="no snapshot store"):
            b.add_adjoint(sid + 7, "elastic", m.data_ptr(), src.data_ptr(), s["ext"], g.data_ptr(), par, s["shape"],
                          (H, H, H))
        b.run()
        assert b.query(sid) == 1 and b.query(12345) == -1
        assert b.status()[0] == 0 and b.status()[1] >= sfp  # the store outlives its forward shot
        with pytest.raises(RuntimeError, match="does not match"):
            b.add_adjoint(sid, "elastic", m.data_ptr(), src.data_ptr(), s["ext"], g.data_ptr(),
                          F.make_param(40, DT, sub=2), s["shape"], (H, H, H))
        b.release(sid)
        assert b.status()[1] == 0
        b.close()
    finally:
        eng.close()


def test_online_tuning_waits_for_a_shot_that_reads_the_chunk():
    """No launch of a one-launch elastic / VTI shot reads the batch's y chunk: a batch of these
    times no candidate; the windows start when an acoustic shot joins, and the traces keep
    their bits through the re-tilings."""
    import torch
    dev = torch.device("cuda:0")
    shots = [make_shot("elastic", (30, 34, 38), 80, 2), make_shot("acoustic", (40, 44, 48), 70, 1)]
    eng = F.Engine(0)
    try:
        b = F.Batch(eng)
        b.autotune(3)
        keep, out = [], []

        def admit(s):
            m, src = torch.from_numpy(s["model"]).to(dev), torch.from_numpy(s["src"]).to(dev)
            r = torch.zeros((F.n_comp(F.PHYSICS[s["physics"]]), s["ext"].npts, s["par"].nt), device=dev)
            torch.cuda.synchronize()
            keep.extend([m, src])
            out.append(r)
            b.add(s["physics"], m.data_ptr(), src.data_ptr(), r.data_ptr(), s["inj"], s["ext"], s["par"], s["shape"],
                  (H, H, H))

        admit(shots[0])
        b.step(20)
        assert b.tiles() == (0, [0.0] * 4)
        admit(shots[1])
        b.run()
        yc, ms = b.tiles()
        assert yc in (4, 8, 16, 32) and all(t > 0 for t in ms)
        b.close()
        for s, r in zip(shots, out):
            assert np.array_equal(r.cpu().numpy(), single(eng, s, dev)), s["physics"]
    finally:
        eng.close()


@pytest.mark.parametrize("physics,shape", [("acoustic", (40, 44, 48)), ("vti", (200, 12, 20))])
def test_shots_hold_the_memory_of_their_step_form(physics, shape):
    """Without the one-launch step a shot holds fields, model, fluxes and small tables, not the
    boundary coefficients (at 384 B per point of a face more than the fluxes on a narrow grid);
    the forward shot of a gradient holds the block that its adjoint takes over."""
    import torch
    dev = torch.device("cuda:0")
    nt = 12
    s = make_shot(physics, shape, nt, 3)
    ny, nx, nz = shape
    cells = ny * nx * ((nz + 63) // 64 * 64)
    fields = {"acoustic": 3 + 2, "elastic": 9 + 3 + 7, "vti": 9 + 7 + 9}[physics] * cells * 4
    fp = F.Batch.footprint(physics, shape, s["inj"], s["ext"])
    assert fp > fields + (1 << 20)
    held = {}
    eng = F.Engine(0)
    try:
        m, src = torch.from_numpy(s["model"]).to(dev), torch.from_numpy(s["src"]).to(dev)
        r = torch.zeros((F.n_comp(F.PHYSICS[physics]), s["ext"].npts, nt), device=dev)
        torch.cuda.synchronize()
        for fused in (False, True):
            eng.tune(fused=fused)
            for sub in (0, 3):
                b = F.Batch(eng)
                b.add(physics, m.data_ptr(), src.data_ptr(), r.data_ptr(), s["inj"], s["ext"],
                      F.make_param(nt, DT, sub=sub), shape, (H, H, H))
                held[fused, sub] = b.status()[1] - (F.Batch.snap_footprint(physics, shape, nt, sub) if sub else 0)
                b.run()
                b.close()
    finally:
        eng.close()
    for sub in (0, 3):
        assert fields <= held[False, sub] <= fields + (64 << 10)  # injector, taper tables and alignment
        assert held[True, sub] == fp
