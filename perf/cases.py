"""What this framework is used for, as timed cases.

A case is a dict of plain values; its "kind" says which use it stands for:

frame    one rendered frame of the reference's demo: the render rank's tunables
         for the frame (its mover moves), four steps, the packed coordinates.
job      a whole small simulation from host particles: upload, step, download.
run      a dam break carried on from a saved state: restore the snapshot, step,
         download.  `settle` steps have been taken before the snapshot, so the
         cases cover the fresh column as well as the compressed pool.  `cap` is
         the reference's bucket cap (0: none).
batch    scenes of uneven sizes and four parameter presets stepped together,
         from a snapshot, and their positions read back.
predict  the learned macro-step's forward pass over a batch of recorded states.
train    one training iteration: sampled states, loss, gradients, Adam.
macro    one judged macro-step from a recorded state, and the positions after it.

Sizes are those of the benchmark and the tests (4,096 and 1,048,576 particles,
256 scenes of 2k-64k, 64 scenes of 16,384, scenes of 65,536), the reference's
demo (1,500), and generic ones between, with lattices that fill no tile.
"""
import math

import numpy as np
import torch

import sph_amd as sa
from sph_amd import scenes as sc
from sph_amd import surrogate as su

SPACING = 0.5   # lattice spacing in units of h, all dam breaks
JITTER = 0.01
LATTICE_NEIGHBOURS = math.pi / SPACING ** 2  # within h at the lattice's density


def listed():
    return [
        # the reference's own scene, one 30 Hz frame: the smallest call there is
        dict(name="frame_1500", kind="frame", n=1500, preset="x"),
        # the 4,096-particle dam break from host memory and back
        dict(name="job_4k", kind="job", nx=64, ny=64, steps=100),
        # small and middle scenes, where a launch does not fill the chip
        dict(name="run_16k", kind="run", nx=127, ny=131, settle=300, steps=64, cap=0),
        dict(name="run_65k", kind="run", nx=256, ny=256, settle=220, steps=64, cap=0),
        # a middle scene that is past the small-scene kernels
        dict(name="run_250k", kind="run", nx=499, ny=503, settle=220, steps=64, cap=0),
        # the same order of size as the reference runs it: 100-slot buckets
        dict(name="run_513k_cap", kind="run", nx=700, ny=733, settle=250, steps=64, cap=100),
        # the headline: the million-particle dam break, early and compressed
        dict(name="run_1m", kind="run", nx=1024, ny=1024, settle=20, steps=200, cap=0),
        dict(name="run_1m_late", kind="run", nx=1024, ny=1024, settle=500, steps=100, cap=0),
        # the batched configuration
        dict(name="batch_256", kind="batch", scenes=256, settle=100, steps=64),
        # the network at its training configuration: forward, one training step
        dict(name="predict_64x16k", kind="predict", scenes=64, n=16384, settle=100),
        dict(name="train_64x16k", kind="train", scenes=64, n=16384, settle=100),
        # judged inference on the wide scenes
        dict(name="macro_16x64k", kind="macro", scenes=16, n=65536, settle=200),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "job", "run", "run", "run", "batch", "predict", "train", "macro"])
    if kind == "frame":
        return dict(kind=kind, n=_log(rng, 500, 20000), preset=rng.choice("xyab"))
    if kind in ("job", "run"):
        n = _log(rng, 2000, 50000 if kind == "job" else 1000000)
        nx = max(8, int(math.sqrt(n) * rng.uniform(0.7, 1.4)))
        ny = max(8, n // nx)
        if kind == "job":
            return dict(kind=kind, nx=nx, ny=ny, steps=rng.randint(20, 120))
        return dict(kind=kind, nx=nx, ny=ny, settle=_log(rng, 10, 500), steps=rng.randint(24, 100),
                    cap=rng.choice([0, 0, 0, 100]))
    if kind == "batch":
        return dict(kind=kind, scenes=_log(rng, 2, 256), settle=_log(rng, 10, 200),
                    steps=rng.randint(8, 48))
    if kind == "macro":
        return dict(kind=kind, scenes=rng.randint(1, 16), n=4 * _log(rng, 1000, 16384),
                    settle=_log(rng, 20, 200))
    return dict(kind=kind, scenes=rng.randint(2, 64), n=_log(rng, 1000, 16384),
                settle=_log(rng, 8, 120))


# --------------------------------------------------------------------------
# inputs


def _dam_break(case, seed):
    """The dam break of the benchmark, its box scaled with the column."""
    nx, ny = case["nx"], case["ny"]
    scale = 1200.0 / 512.0
    return sc.dam_break(nx, ny, (nx * SPACING * scale, ny * SPACING * 800.0 / 512.0), seed=seed + 1)


def _slosh_scenes(case, seed):
    """Sloshing dam breaks of n particles each, boxes with the training
    scenes' proportions; four times as wide for the judged macro-step."""
    n, widen = case["n"], 4 if case["kind"] == "macro" else 1
    side = math.sqrt(n / widen / 16384.0)
    return sc.sloshing_dam_breaks(case["scenes"], n=n, box=(128.0 * side * widen, 96.0 * side),
                                  seed=seed + 1, widen=widen)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        tun, box, parts, info = sc.reference_scene(case["preset"], n_global=case["n"])
        # the demo's lattice with the seed's small displacements
        rng = np.random.default_rng(seed)
        for f in ("x", "y"):
            d = rng.uniform(-0.01, 0.01, len(parts)) * info["spacing"]
            parts[f] = np.maximum(parts[f] + d, 0).astype(np.float32)
        frames = []
        for cx, cy in sc.attract_mover_path(None, box, 64, gl_x0=rng.uniform(-0.9, 0.3)):
            t = sa.Tunables.from_buffer_copy(bytes(tun))
            t.mover_center_x, t.mover_center_y = float(cx), float(cy)
            frames.append(t)
        s = sa.Solver(frames[0], box, info["capacity"])
        s.set_bucket_cap()
        s.upload(parts)
        s.step(32)
        s.sync()
        return dict(case=case, solver=s, frames=frames, at=0)
    if kind == "job":
        tun, box, parts = _dam_break(case, seed)
        s = sa.Solver(tun, box, len(parts))
        s.upload(parts)
        s.step(2)
        s.sync()
        return dict(case=case, solver=s, parts=parts)
    if kind == "run":
        tun, box, parts = _dam_break(case, seed)
        s = sa.Solver(tun, box, len(parts))
        s.set_bucket_cap(case["cap"])
        s.upload(parts)
        s.step(max(2, case["settle"]))
        s.snapshot_save()
        s.sync()
        return dict(case=case, solver=s)
    if kind == "batch":
        # the benchmark's scene sizes and boxes, the particles moved by the seed
        scenes = sc.batched_scenes(case["scenes"])
        parts, counts = sc.concat(scenes)
        rng = np.random.default_rng(seed)
        for f in ("x", "y"):
            parts[f] += rng.uniform(-JITTER, JITTER, len(parts)).astype(np.float32)
        s = sa.Solver.batch([(t, b, len(p)) for t, b, p, _ in scenes])
        s.upload_batch(parts, counts)
        s.step(max(2, case["settle"]))
        s.snapshot_save()
        s.sync()
        return dict(case=case, solver=s)
    # the learned macro-step: two recorded frames, four steps apart
    scenes = _slosh_scenes(case, seed)
    s = su.make_batch(scenes)
    tr = sa.Trajectory(len(scenes), case["n"], 2)
    s.step(max(2, case["settle"]))
    tr.record(s, 0)
    s.step(su.MACRO)
    tr.record(s, 1)
    model = sa.Surrogate(seed=seed + 1)
    if kind != "train":
        su.load_weights(model)
    which = np.arange(len(scenes), dtype=np.int32)
    st = dict(case=case, solver=s, traj=tr, model=model, scenes=scenes, which=which,
              first=np.zeros(len(scenes), np.int32))
    for k in range(len(scenes)):
        s.set_scene_time_offset(k, max(2, case["settle"]))
    _recorded_state(st)
    if kind == "macro":  # the judge's first macro-steps, which set its references up
        for _ in range(2):
            model.macro_step(s, 0.01)
            _recorded_state(st)
    s.sync()
    return st


def _recorded_state(st):
    st["traj"].load(st["solver"], st["which"], st["first"])
    st["solver"].phase("hash")


# --------------------------------------------------------------------------
# one pass


def _whole(p):
    """Particle records as numbers: the 12 float fields, and the ids."""
    return {"fields": p.view(np.float32).reshape(-1, 13)[:, :12], "id": p["id"]}


def run(st):
    case, s = st["case"], st["solver"]
    kind = case["kind"]
    if kind == "frame":
        st["at"] = (st["at"] + 1) % len(st["frames"])
        s.set_tunables(st["frames"][st["at"]])
        s.step(sc.REFERENCE_STEPS_PER_FRAME)
        return s.pack_coords()
    if kind == "job":
        s.upload(st["parts"])
        s.step(case["steps"])
        return _whole(s.download())
    if kind == "run":
        s.snapshot_restore([1])
        s.step(case["steps"])
        return _whole(s.download())
    if kind == "batch":
        s.snapshot_restore([1] * case["scenes"])
        s.step(case["steps"])
        return s.download_positions()
    _recorded_state(st)
    model = st["model"]
    if kind == "predict":
        return model.predict(s)
    if kind == "train":
        model.zero_grads()
        loss = model.backward_trajectory(s, st["traj"])
        grads = model.grads()
        model.adam(1e-3)
        return {"loss": loss, "grads": grads}
    flags = model.macro_step(s, 0.01)
    return {"flags": flags, "xy": s.download_positions()}


# --------------------------------------------------------------------------
# the work of a pass


def _step_work(n, cells, steps):
    """A step's compulsory traffic by phase, and its pair terms at the
    lattice's neighbour count (three passes, about 25 operations each)."""
    return {"bytes": steps * (192.0 * n + 56.0 * cells),
            "flops": steps * n * 3 * LATTICE_NEIGHBOURS * 25.0}


def _network_work(n, backward):
    """Per particle: the edge layer over its neighbours (6 -> 64 and the
    activation), then 64 -> 64, 69 -> 64 and 64 -> 2 per particle."""
    edge = LATTICE_NEIGHBOURS * (2 * 6 * 64 + 4 * 64)
    node = 2 * 64 * 64 + 2 * 69 * 64 + 2 * 2 * 64
    return {"bytes": n * (16.0 + 8.0 + (8.0 if backward else 0.0)),
            "flops": n * (edge + node) * (3.0 if backward else 1.0)}


def work(case):
    kind = case["kind"]
    if kind == "frame":
        n = case["n"]
        w = _step_work(n, n / 4, sc.REFERENCE_STEPS_PER_FRAME)
        return {"bytes": w["bytes"] + 4.0 * n, "flops": w["flops"]}
    if kind in ("job", "run"):
        n = case["nx"] * case["ny"]
        w = _step_work(n, n * 960000.0 / 1048576.0, case["steps"])
        return {"bytes": w["bytes"] + 52.0 * n * (2 if kind == "job" else 1), "flops": w["flops"]}
    if kind == "batch":
        # sizes are log-uniform in [2048, 65536]; cells = area / h^2 with the
        # fluid filling 0.2-0.5 of the box
        n = case["scenes"] * (65536 - 2048) / math.log(65536 / 2048)
        w = _step_work(n, n * SPACING ** 2 / 0.33, case["steps"])
        return {"bytes": w["bytes"] + 8.0 * n, "flops": w["flops"]}
    n = case["scenes"] * case["n"]
    if kind in ("predict", "train"):
        return _network_work(n, kind == "train")
    # network and judge over every scene, four plain steps over the scheduled
    # sixteenth of them
    a, b = _network_work(n, False), _step_work(n, 0.75 * n, 4 / 16)
    return {"bytes": a["bytes"] + b["bytes"] + 48.0 * n, "flops": a["flops"] + b["flops"]}


# --------------------------------------------------------------------------
# the network in 64 bits


def _edges(x, h):
    """All ordered pairs (i, j), i != j, of one scene within h."""
    out = []
    for lo in range(0, len(x), 1024):
        d2 = ((x[lo:lo + 1024, None, :] - x[None, :, :]) ** 2).sum(-1)
        i, j = torch.nonzero(d2 <= h * h, as_tuple=True)
        i = i + lo
        out.append(torch.stack([i[i != j], j[i != j]]))
    return torch.cat(out, 1)


def _network(p, x, v, e, h, dt, ax, ay):
    """Displacements over four steps of one scene, in 64 bits."""
    W1, W2 = p[:1024].view(64, 16)[:, :6], p[1024:5120].view(64, 64)
    b2, W3 = p[5120:5184], p[5184:10304].view(64, 80)[:, :69]
    W4, b4 = p[10304:10432].view(2, 64), p[10432:10434]
    i, j = e
    d, dv = (x[j] - x[i]) / h, (v[j] - v[i]) * 0.2
    f = torch.cat([d, dv, d.norm(dim=1, keepdim=True), torch.ones_like(d[:, :1])], 1)
    S = torch.zeros(len(x), 64, dtype=x.dtype, device=x.device)
    S = S.index_add(0, i, torch.nn.functional.silu(f @ W1.T))
    deg = torch.bincount(i, minlength=len(x)).to(x.dtype)
    m = S @ W2.T + deg[:, None] * b2
    a = torch.tensor([ax, ay], dtype=x.dtype, device=x.device)
    u = torch.cat([m, 0.2 * v, (0.1 * a).expand(len(x), 2), torch.ones_like(x[:, :1])], 1)
    out = torch.nn.functional.silu(u @ W3.T) @ W4.T + b4
    return 4 * dt * v + 10 * dt * dt * a + 0.05 * out


def exact(case, seed):
    """The network's outputs in 64 bits for the recorded states.  A run of
    many steps has no such value: the flow is chaotic, and 32 and 64 bits are
    different flows after a few dozen steps."""
    kind = case["kind"]
    if kind not in ("predict", "train") or case["scenes"] * case["n"] ** 2 > 3e10:
        return None
    st = prepare(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    a, b = (torch.from_numpy(st["traj"].read(f)).to(dev, torch.float64) for f in (0, 1))
    p = torch.from_numpy(st["model"].params).to(dev, torch.float64)
    p.requires_grad_(kind == "train")
    pred, loss = [], 0.0
    for k, (tun, _, _, amp, period) in enumerate(st["scenes"]):
        h, dt = float(tun.smoothing_radius), float(tun.time_step)
        t = max(2, case["settle"]) * dt
        ax = -amp * math.sin(2 * math.pi / period * t)
        x, v = a[k, :, :2], a[k, :, 2:]
        d = _network(p, x, v, _edges(x, h), h, dt, ax, -float(tun.g))
        if kind == "train":
            part = (((d - (b[k, :, :2] - x)) / 0.05) ** 2).sum() / (case["scenes"] * case["n"])
            part.backward()
            loss += float(part.detach())
        else:
            pred.append(d)
    if kind == "train":
        return {"loss": loss, "grads": p.grad.cpu().numpy()}
    return torch.cat(pred).cpu().numpy()
