"""The work a program using this library has it do, as measurable cases.

Every case goes through a public entry point: a scene's substeps
(``apbf_amd.scene.Scene`` / ``PackedBatch``), one substep over caller-owned
device lists (``apbf_amd.lists.pool_update``), a list operator
(``apbf_amd.ops``) or the warm-start network (``apbf_amd.learned``).

A simulation case steps from a keyframe: a pass puts the keyframe back (the
time machine's jump, or the caller's own copy of its lists), steps, and reads
the state the steps leave. So a pass can be repeated, and every pass does the
same work. Scenes are read to the host, as a program that shows or stores them
does, into the pinned buffers it keeps for that; lists stay on the device, in
the buffers of the caller. Both are as long as the capacities.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from apbf_amd import _lib, config, learned, lists, ops
from apbf_amd.scene import PackedBatch, Scene

DT = 1.0 / 120.0
FIXED = 262144.0  # position units per world unit


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # The reference's default build and scene: the planar pool (40 x 20
        # particles), binary-search neighbourhood, 60 substeps a second, drawn
        # every fourth. The smallest scene: its time is launches and latency.
        dict(name="planar_pool_800", kind="scene", scene="pool2d", radius=1.0, method="binary_search", steps=4,
             graph=False),
        # The reference's pool in 3D (16 000 particles, adaptive, kernel widths
        # from boundary distances, hash grid), drawn every fourth substep.
        dict(name="pool_16000", kind="scene", scene="pool3d", radius=1.0, method="green", steps=4, graph=False),
        # The plain dam break of 32^3 particles, 3 iterations, replayed from a
        # captured graph as a serving loop does.
        dict(name="dam_break_32768_graph", kind="scene", scene="dam_break", side=32, method="green", steps=16,
             graph=True),
        # An adaptive water drop of ordinary size with ragged counts: kernel
        # width spreading, splits and merges, 4 iterations.
        dict(name="water_drop_43k", kind="scene", scene="drop", px=47, py=19, pz=43, drop=5001, method="green",
             steps=8, graph=False),
        # The 1.1 M-particle adaptive water drop from rest, the framework's
        # headline workload: 12 substeps (a tenth of a second), then the state.
        dict(name="settled_drop_1100k", kind="scene", scene="settled", px=180, py=50, pz=180, drop=100000,
             settle=200, method="green", steps=12, graph=False),
        # The large uniform pool at rest density (8 M particles, plain PBF,
        # 3 iterations) over the caller's own device lists, two substeps.
        dict(name="large_pool_8m_lists", kind="lists", scene="large_pool", nx=386, ny=107, nz=193, steps=2),
        # An adaptive drop over caller-owned lists, one operator per stage.
        dict(name="water_drop_230k_lists", kind="lists", scene="drop", px=91, py=25, pz=89, drop=25000, steps=2),
        # Sixteen independent scenes (plain dam breaks and adaptive drops) as
        # packed lists, one launch per stage for all of them.
        dict(name="batch_16_scenes", kind="batch", count=16, n_min=5000, n_max=60000, steps=8),
        # The list algorithm every neighbourhood build starts with, called on
        # its own: a stable sort of 18-bit cell hashes with their particle ids.
        dict(name="sort_1m_18bit", kind="sort", n=1000003, bits=18),
        # The warm-start network over every particle of the headline drop.
        dict(name="mlp_forward_1100k", kind="mlp_forward", n=1122976),
        # Its training direction: loss and gradient over a harvested batch.
        dict(name="mlp_gradient_260k", kind="mlp_gradient", n=262147),
        # Harvesting (feature, lambda) pairs from plain substeps, the input of
        # the network's training.
        dict(name="harvest_120k", kind="harvest", scene="drop", px=71, py=23, pz=67, drop=12000, steps=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drop_sizes(rng, lo, hi):
    n = _log(rng, lo, hi)
    px = max(8, int(round((0.9 * n / 0.27) ** (1.0 / 3.0) * rng.uniform(0.9, 1.1))))
    pz = max(8, int(round((0.9 * n / 0.27) ** (1.0 / 3.0) * rng.uniform(0.9, 1.1))))
    return dict(px=px, py=max(4, int(round(0.9 * n / (px * pz)))), pz=pz, drop=max(200, n // 10 + rng.randrange(7)))


def draw(rng):
    kind = rng.choice(["pool2d", "pool3d", "dam_break", "drop", "drop", "settled", "large_pool", "drop_lists", "batch",
                       "sort", "mlp_forward", "mlp_gradient", "harvest"])
    if kind == "pool2d":
        return dict(kind="scene", scene=kind, radius=round(math.exp(rng.uniform(math.log(0.2), math.log(1.0))), 3),
                    method=rng.choice(["binary_search", "green"]), steps=rng.randrange(2, 9), graph=rng.random() < 0.3)
    if kind == "pool3d":
        return dict(kind="scene", scene=kind, radius=round(rng.uniform(0.4, 1.3), 3), method="green",
                    steps=rng.randrange(2, 7), graph=rng.random() < 0.3)
    if kind == "dam_break":
        return dict(kind="scene", scene=kind, side=_log(rng, 12, 72), method="green", steps=2 * rng.randrange(2, 9),
                    graph=rng.random() < 0.6)
    if kind == "drop":
        return dict(kind="scene", scene=kind, method="green", steps=2 * rng.randrange(2, 5),
                    graph=rng.random() < 0.3, **_drop_sizes(rng, 8000, 400000))
    if kind == "settled":
        a = rng.randrange(60, 170)
        return dict(kind="scene", scene=kind, px=a, py=rng.randrange(20, 50), pz=rng.randrange(60, 170),
                    drop=_log(rng, 3000, 80000), settle=rng.randrange(20, 200), method="green", steps=rng.randrange(6, 13), graph=False)
    if kind == "large_pool":
        nx, nz = _log(rng, 60, 380), _log(rng, 40, 190)
        return dict(kind="lists", scene=kind, nx=nx, ny=_log(rng, 20, 105), nz=nz, steps=rng.randrange(1, 3))
    if kind == "drop_lists":
        return dict(kind="lists", scene="drop", steps=rng.randrange(1, 4), **_drop_sizes(rng, 8000, 400000))
    if kind == "batch":
        return dict(kind=kind, count=rng.randrange(4, 17), n_min=5000, n_max=_log(rng, 20000, 80000),
                    steps=rng.randrange(2, 9))
    if kind == "sort":
        return dict(kind=kind, n=_log(rng, 1000, 8000000), bits=rng.choice([12, 15, 18, 21, 24, 30, 32]))
    if kind in ("mlp_forward", "mlp_gradient"):
        return dict(kind=kind, n=_log(rng, 1000, 4000000 if kind == "mlp_forward" else 1000000))
    return dict(kind="harvest", scene="drop", steps=rng.randrange(2, 4), **_drop_sizes(rng, 8000, 400000))


# ------------------------------------------------------------------ the inputs
def _scene_inputs(case, seed):
    """(params, state) of a case's scene. Seeds move every particle: the
    lattices are jittered (the reference's pools start unjittered, so theirs
    are moved by up to 2 % of the radius here)."""
    kind = case["scene"]
    if kind in ("pool2d", "pool3d"):
        p, st = config.pool_scene(radius=case["radius"], dims=2 if kind == "pool2d" else 3)
        rng = np.random.default_rng(seed)
        axes = 2 if kind == "pool2d" else 3
        m = int(0.02 * case["radius"] * FIXED)
        st["position"][:, :axes] += rng.integers(-m, m + 1, (len(st["radius"]), axes), dtype=np.int32)
        st["pos_backup"] = st["position"].copy()
        p["dt"] = 1.0 / 60.0
        return p, st
    if kind == "dam_break":
        return config.dam_break(n_side=case["side"], seed=seed)
    if kind == "drop":
        return config.water_drop(pool_counts=(case["px"], case["py"], case["pz"]), drop_particles=case["drop"],
                                 seed=seed, res=5 if case["px"] < 64 else 6, pairs_per_particle=400)
    if kind == "settled":
        p, st, _ = config.settled_water_drop(pool_counts=(case["px"], case["py"], case["pz"]),
                                             drop_particles=case["drop"], settle=case["settle"], drop_settle=20,
                                             seed=seed)
        # capacities by the lattice it came from, so they do not depend on the seed
        p["cap_particles"] = case["px"] * case["py"] * case["pz"] + case["drop"]
        p["cap_pairs"] = p["cap_particles"] * 800
        p["cap_transfers"] = p["cap_particles"] // 4
        return p, st
    raise ValueError(kind)


def _large_pool_lists(case, seed):
    """The large pool at rest density (config.large_pool), its state made on
    the device: a lattice of nx x ny x nz particles of radius h/4 at 2.068
    radii, jittered by 0.01 h, the slab x < 20 h moving at 4 h/s."""
    r, spacing = 0.25, 2.068 * 0.25
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    box = (max(20.0, (nx + 1) * spacing), max(20.0, 2.0 * ny * spacing), max(20.0, (nz + 1) * spacing))
    p, _ = config.large_pool(box=box, n_target=1000)
    # cells of about 0.78 h, as the full-size pool's
    p["hash_res_log2"] = min(8, max(3, int(math.floor(math.log2(max(box) / 0.75)))))
    p["cap_particles"], p["cap_pairs"] = n, n * 128
    g = torch.Generator(device="cuda").manual_seed(seed)
    i = torch.arange(n, device="cuda")
    at = torch.stack([i // (ny * nz), (i // nz) % ny, i % nz], 1).to(torch.float64)
    at = (at + 0.5) * spacing + (torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64) - 0.5) * 0.02
    q = lists.ParticleLists(n)
    q.position[:, :3] = (at * FIXED).to(torch.int32)
    q.pos_backup.copy_(q.position)
    q.pos_backup[:, 0] -= (at[:, 0] < 20.0).to(torch.int32) * int(4.0 * DT * FIXED)
    q.radius.fill_(r)
    q.inverse_mass.fill_(1.0 / (2.0 * r) ** 3)
    q.target_radius.fill_(r)
    q.kernel_width.fill_(4.0 * r)
    q.boundariness.fill_(1.0)
    q.boundary_distance.fill_(int(r * FIXED))
    q.length.fill_(n)
    return p, q, lists.TransferLists(p["cap_transfers"])


def _batch_scenes(case, seed):
    """config.batch_scenes, with the particle counts spread evenly over the
    logarithm of the range: plain dam breaks and adaptive drops in turn."""
    out = []
    for k in range(case["count"]):
        n = case["n_min"] * (case["n_max"] / case["n_min"]) ** ((k + 0.5) / case["count"])
        if k % 2 == 0:
            out.append(config.dam_break(n_side=max(4, int(round(n ** (1.0 / 3.0)))), seed=seed + k))
        else:
            a = max(6, int(round((0.9 * n / 0.27) ** (1.0 / 3.0))))
            out.append(config.water_drop(pool_counts=(a, max(3, int(round(0.27 * a))), a), seed=seed + k, res=5,
                                         drop_particles=max(100, int(n) // 10), pairs_per_particle=300,
                                         target_scale=0.05))
    return out


def _network(seed):
    """He-initialised weights of the 16-64-64-1 network and its normalisation."""
    rng = np.random.default_rng(seed)
    w = np.concatenate([rng.standard_normal(1024) * math.sqrt(2.0 / 16), rng.standard_normal(64) * 0.05,
                        rng.standard_normal(4096) * math.sqrt(2.0 / 64), rng.standard_normal(64) * 0.05,
                        rng.standard_normal(64) * math.sqrt(1.0 / 64), [0.02]]).astype(np.float32)
    norm = np.concatenate([rng.standard_normal(16), rng.uniform(0.3, 3.0, 16), [0.7]]).astype(np.float32)
    return w, norm


def _samples(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((case["n"], 16), generator=g, device="cuda")
    t = torch.randn(case["n"], generator=g, device="cuda")
    return x, t


def _sort_inputs(case, seed):
    """Cell hashes of particles that fill a part of the grid: every particle
    of a cell has the same key, and the cells come nearly sorted in runs, as
    after the previous substep's sort."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, top = case["n"], 1 << case["bits"]
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    at = (torch.arange(n, device="cuda", dtype=torch.float64) / n + 0.02 * (u - 0.5)).clamp(0.0, 1.0 - 1e-9)
    some = torch.rand(n, generator=g, device="cuda") < 0.1
    keys = (torch.where(some, u, at) * top).to(torch.int64)
    keys = torch.where(keys >= 1 << 31, keys - (1 << 32), keys).to(torch.int32)
    return keys, torch.arange(n, dtype=torch.int32, device="cuda")


class _Keyframe:
    """A scene's keyframe (apbf_snapshot)."""

    def __init__(self, scene):
        self._L, self._scene, self._h = _lib.lib(), scene, C.c_void_p()
        _lib.check(self._L.apbf_snapshot_create(scene._h, C.byref(self._h)), "apbf_snapshot_create")

    def load(self):
        _lib.check(self._L.apbf_snapshot_restore(self._h, self._scene._h), "apbf_snapshot_restore")

    def __del__(self):
        self._L.apbf_snapshot_destroy(self._h)


class _Readback:
    """A scene's state on the host (apbf_scene_get_state without the pairs), in
    pinned buffers of the scene's capacities."""

    def __init__(self, scene, p):
        def pinned(n, dtype):
            return torch.zeros(n, dtype=dtype, pin_memory=True)

        n, nt = int(p["cap_particles"]), int(p["cap_transfers"])
        i, f = torch.int32, torch.float32
        self._L, self._scene = _lib.lib(), scene
        self.out = dict(position=pinned((n, 4), i), velocity=pinned((n, 4), f), inverse_mass=pinned(n, f),
                        radius=pinned(n, f), pos_backup=pinned((n, 4), i), transferring=pinned(n, i),
                        target_radius=pinned(n, f), kernel_width=pinned(n, f), boundariness=pinned(n, f),
                        boundary_distance=pinned(n, i), t_source=pinned(nt, i), t_target=pinned(nt, i),
                        t_time_left=pinned(nt, f))

    def read(self):
        at = [C.c_void_p(v.data_ptr()) for v in self.out.values()]
        last_dt = C.c_float()
        _lib.check(self._L.apbf_scene_get_state(self._scene._h, *at, None, C.byref(last_dt)), "apbf_scene_get_state")
        return self.out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("scene", "harvest"):
        p, st = _scene_inputs(case, seed)
        scene = Scene(p)
        scene.set_state(st)
        if kind == "scene":
            scene.set_neighborhood_method(case["method"])
            if case["graph"]:
                scene.capture(p["dt"])
        state = dict(case=case, scene=scene, key=_Keyframe(scene), dt=p["dt"])
        if kind == "scene":
            state["readback"] = _Readback(scene, p)
        else:  # harvested rows: one per particle and substep
            m = p["cap_particles"] * (case["steps"] - 1)
            state["features"], state["targets"] = torch.zeros((m, 16), device="cuda"), torch.zeros(m, device="cuda")
        return state
    if kind == "lists":
        if case["scene"] == "large_pool":
            p, q, t = _large_pool_lists(case, seed)
            last_dt = DT
        else:
            p, st = _scene_inputs(case, seed)
            q = lists.ParticleLists.from_state(st, p["cap_particles"])
            t = lists.TransferLists(p["cap_transfers"], st=st)
            last_dt = st["last_delta_time"]
        nb = lists.NeighborLists(p["cap_particles"], p["cap_pairs"])
        fields = ("position", "velocity", "pos_backup") + q.F32 + q.U32
        out = {k: torch.zeros_like(getattr(q, k)) for k in fields}
        out.update({"t_" + k: torch.zeros_like(getattr(t, k)) for k in ("source", "target", "time_left")})
        out.update({k: torch.zeros_like(getattr(nb, k)) for k in ("row_offset", "neighbors")})
        return dict(case=case, ctx=lists.Context(p), q=q, t=t, nb=nb, dt=p["dt"], last_dt=last_dt, out=out,
                    key={k: getattr(q, k).clone() for k in fields + ("length",)}, t_len=t.length.clone())
    if kind == "batch":
        cases = _batch_scenes(case, seed)
        batch = PackedBatch(cases)
        return dict(case=case, batch=batch, keys=[_Keyframe(g["scene"]) for g in batch.groups], dt=DT,
                    readbacks=[_Readback(g["scene"], g["scene"].params) for g in batch.groups])
    if kind == "sort":
        keys, ids = _sort_inputs(case, seed)
        return dict(case=case, keys=keys, ids=ids)
    w, norm = _network(seed)
    x, t = _samples(case, seed)
    return dict(case=case, model=learned.WarmStartModel(w, norm), x=x, t=t)


# -------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "scene":
        scene = state["scene"]
        state["key"].load()
        if case["graph"]:
            scene.replay(case["steps"] // 2)
        else:
            for _ in range(case["steps"]):
                scene.update(state["dt"])
        return state["readback"].read()
    if kind == "harvest":
        state["key"].load()
        f, t = learned.harvest(state["scene"], case["steps"], state["dt"])
        learned.set_mode(state["scene"], None, "off")
        state["features"][:f.shape[0]] = f
        state["targets"][:t.shape[0]] = t
        return state["features"], state["targets"]
    if kind == "lists":
        q, t, nb, ctx, out = state["q"], state["t"], state["nb"], state["ctx"], state["out"]
        for k, v in state["key"].items():
            getattr(q, k).copy_(v)
        t.length.copy_(state["t_len"])
        ctx.last_delta_time.value = state["last_dt"]
        for _ in range(case["steps"]):
            lists.pool_update(ctx, q, t, nb, state["dt"])
        n, nt = q.n(), int(t.length.item())
        rows, pairs = int(nb.rows.item()), int(nb.length.item())
        used = dict(t_source=(t.source, nt), t_target=(t.target, nt), t_time_left=(t.time_left, nt),
                    row_offset=(nb.row_offset, rows + 1), neighbors=(nb.neighbors, pairs))
        for k, v in out.items():  # what the lists hold, into the caller's buffers
            src, m = used[k] if k in used else (getattr(q, k), n)
            v[:m] = src[:m]
        return out
    if kind == "batch":
        for k in state["keys"]:
            k.load()
        for _ in range(case["steps"]):
            state["batch"].update(state["dt"])
        return [r.read() for r in state["readbacks"]]
    if kind == "sort":
        return ops.radix_sort(state["keys"], state["ids"],
                              upper_bound=min((1 << case["bits"]) - 1, 0xFFFFFFFF))
    if kind == "mlp_forward":
        return state["model"].forward(state["x"])
    return state["model"].gradient(state["x"], state["t"])


# ------------------------------------------------------------ what it takes
def _particles(case):
    kind = case.get("scene", case["kind"])
    if kind == "pool2d":
        return int(80 / (2 * case["radius"])) * int(40 / (2 * case["radius"]))
    if kind == "pool3d":
        return int(80 / (2 * case["radius"])) * int(40 / (2 * case["radius"])) ** 2
    if kind == "dam_break":
        return case["side"] ** 3
    if kind == "drop":
        return case["px"] * case["py"] * case["pz"] + case["drop"]
    if kind == "settled":
        return int(0.63 * case["px"] * case["py"] * case["pz"] + 0.88 * case["drop"])
    if kind == "large_pool":
        return case["nx"] * case["ny"] * case["nz"]
    a, b = math.log(case["n_min"]), math.log(case["n_max"])  # batch: the mean of a log-uniform draw
    return int(case["count"] * (case["n_max"] - case["n_min"]) / max(b - a, 1e-9))


# mean neighbours per particle of the solver's list and of the search, and
# solver iterations, of each kind of scene
_PAIRS = {"pool2d": (12, 12, 3), "pool3d": (32, 32, 3), "dam_break": (26, 26, 3), "drop": (70, 90, 4),
          "settled": (61, 202, 4), "large_pool": (26, 26, 3), "batch": (45, 55, 3)}


def work(case):
    """Simulations: the particle state (88 B) in and out once per substep, and
    per solver pair and iteration about 70 floating-point operations (the
    kernel, its gradient, five sums, the shift), per searched pair 18 (two
    distance tests). A sort: keys and values in and out once. The network:
    2 * 5 184 operations a sample, three times that for the gradient."""
    kind, n = case["kind"], case.get("n")
    if kind == "sort":
        return dict(bytes=16.0 * n, flops=0.0)
    if kind == "mlp_forward":
        return dict(bytes=68.0 * n, flops=2.0 * 5184 * n)
    if kind == "mlp_gradient":
        return dict(bytes=68.0 * n, flops=6.0 * 5184 * n)
    n = _particles(case)
    kept, found, iterations = _PAIRS[case.get("scene", kind)]
    each = n * (70.0 * kept * iterations + 18.0 * found)
    return dict(bytes=176.0 * n * case["steps"], flops=each * case["steps"])


# ------------------------------------------------------------------ in 64 bits
def exact(case, seed):
    """The substeps work on positions of 2^-18 units with truncated sums and
    have no 64-bit counterpart; the network has one, and the sort is exact."""
    kind = case["kind"]
    if kind == "sort":
        keys, ids = _sort_inputs(case, seed)
        order = torch.sort(keys.to(torch.int64) & 0xFFFFFFFF, stable=True).indices
        return keys[order], ids[order]
    if kind not in ("mlp_forward", "mlp_gradient"):
        return None
    w, norm = (torch.from_numpy(a.astype(np.float64)).cuda() for a in _network(seed))
    x, t = _samples(case, seed)
    w1, b1, w2 = w[:1024].view(64, 16), w[1024:1088], w[1088:5184].view(64, 64)
    b2, w3, b3 = w[5184:5248], w[5248:5312], w[5312]
    n = case["n"]
    out = torch.empty(n, dtype=torch.float64, device="cuda")
    grad = torch.zeros(5313, dtype=torch.float64, device="cuda")
    loss = 0.0
    for a in range(0, n, 1 << 18):
        xn = (x[a:a + (1 << 18)].double() - norm[:16]) * norm[16:32]
        z1 = xn @ w1.t().contiguous() + b1
        h1 = z1.clamp_min(0.0)
        z2 = h1 @ w2.t().contiguous() + b2
        h2 = z2.clamp_min(0.0)
        y = h2 @ w3 + b3
        out[a:a + (1 << 18)] = y * norm[32]
        if kind == "mlp_forward":
            continue
        d = y - t[a:a + (1 << 18)].double() / norm[32]
        loss += float(0.5 * (d * d).sum()) / n
        dy = d / n
        dz2 = dy[:, None] * w3[None, :] * (z2 > 0)
        dz1 = (dz2 @ w2) * (z1 > 0)
        grad += torch.cat([(dz1.t().contiguous() @ xn).reshape(-1), dz1.sum(0),
                           (dz2.t().contiguous() @ h1).reshape(-1), dz2.sum(0), h2.t().contiguous() @ dy,
                           dy.sum()[None]])
    return out if kind == "mlp_forward" else (grad.cpu().numpy(), loss)
