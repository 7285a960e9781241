"""Timed cases of the BP inference path, through the package's public calls.

A case is a dict of plain values; ``listed()`` names the standing ones,
``draw(rng)`` gives further ones of the same ranges.  ``prepare(case, seed)``
makes what a program holds before the call (keyframes of a synthetic scene,
and for the kinds that keep one, a context), ``run(state)`` is one pass,
``work(case)`` an estimate of what the pass cannot do without, and
``exact(case, seed)`` the outputs in 64 bits, computed with torch alone.

Kinds:
  build   a map from scratch: context, keyframes, BP, bricks and marginals
  refine  more BP iterations on a context that is kept, marginals read back
  online  keyframes arriving one by one, BP after each, marginals at the end
  repose  one keyframe of a kept context moved (a corrected pose), BP, marginals
  load    an external occupancy map loaded and scored from one frame
  score   a BP map scored from its keyframes (likelihood, depth, accuracy)
  train   the warm start's network trained on voxel features
"""
import math

import numpy as np
import torch

from mrfmap_amd import GVDBInference, GVDBMapLikelihoodEstimator, _lib, gvdb_params, synth

F_EPS = 1e-4
# scene extents (m) and rough planar ray lengths (m) of the two synthetic rooms
DIMS = {"room": (4.0, 4.0, 3.0), "large": (10.0, 10.0, 3.0)}
RAY_M = {"room": 2.6, "large": 5.5}
UNEVEN = ((240, 320), (480, 640), (480, 848))


def listed():
    room = {"scene": "room", "activation": "full", "vis": "brick", "focal": 0.82}
    return [
        # the smallest call: a live 4-keyframe map at 4 cm, refined by 5 iterations
        dict(room, name="refine-qqvga-4cm", kind="refine", rows=120, cols=160, frames=4, res=0.04, iters=5),
        # the same map from nothing: context, lists, launches and readback of a small job
        dict(room, name="build-qqvga-4cm", kind="build", rows=120, cols=160, frames=4, res=0.04, iters=5),
        # a mapper at work: each new 320x240 keyframe is followed by a 3-iteration call
        dict(room, name="online-qvga-2cm", kind="online", rows=240, cols=320, frames=6, res=0.02, iters=3),
        # the reference's own configuration: 2 cm, endpoint activation, sigma 5 cm, 3 iterations
        dict(room, name="build-vga-endpoint", kind="build", rows=480, cols=640, frames=7, res=0.02, iters=3,
             activation="endpoint", focal=0.5959, sigma=0.05),
        # the benchmark's 13 keyframes at 1 cm, mapped from nothing
        dict(room, name="build-vga-1cm", kind="build", rows=480, cols=640, frames=13, res=0.01, iters=3),
        # the same map iterated on: the steady state of a converging map
        dict(room, name="refine-vga-1cm", kind="refine", rows=480, cols=640, frames=13, res=0.01, iters=20),
        # an odd image size and voxel size, with the visibility carried along the ray
        dict(room, name="refine-ragged-carry", kind="refine", rows=315, cols=427, frames=5, res=0.015, iters=10,
             vis="carry"),
        # uneven keyframes of three cameras in a large room: many pairs per update
        dict(room, name="refine-uneven-large", kind="refine", scene="large", rows=0, cols=0, frames=10, res=0.01,
             iters=3),
        # a loop closure moves one keyframe of six
        dict(room, name="repose-vga-1cm", kind="repose", rows=480, cols=640, frames=6, res=0.01, iters=3),
        # an OctoMap-like map brought in and scored against one depth frame
        dict(room, name="load-vga-2cm", kind="load", rows=480, cols=640, frames=1, res=0.02, iters=0),
        # a finished map scored from every keyframe
        dict(room, name="score-vga-1cm", kind="score", rows=480, cols=640, frames=4, res=0.01, iters=3),
        # the warm start's network: two epochs of Adam on a map's worth of samples
        {"name": "train-150k", "kind": "train", "n": 150001, "batch": 8192, "epochs": 2},
    ]


def _updates(case):
    """Rough (ray, voxel) incidences of all keyframes."""
    pix = case["rows"] * case["cols"] or sum(r * c for r, c in UNEVEN) / len(UNEVEN)
    return case["frames"] * pix * RAY_M[case["scene"]] / case["res"] * 1.45


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("build", "refine", "refine", "online", "repose", "load", "score", "train"))
    if kind == "train":
        return {"kind": kind, "n": int(_log_uniform(rng, 3000, 200000)), "batch": rng.choice((2048, 4096, 8192)),
                "epochs": rng.randint(1, 3)}
    while True:
        rows = int(_log_uniform(rng, 96, 480))
        cols = int(rows * rng.uniform(1.2, 1.5))
        case = {"kind": kind, "scene": rng.choice(("room", "room", "large")), "rows": rows, "cols": cols,
                "frames": rng.randint(2, 8), "res": round(_log_uniform(rng, 0.01, 0.04), 4),
                "iters": rng.choice((1, 2, 3, 3, 5, 10)), "focal": round(rng.uniform(0.55, 0.95), 3),
                "activation": rng.choice(("full", "full", "endpoint")), "vis": rng.choice(("brick", "brick", "carry"))}
        if kind == "load":
            case.update(frames=1, iters=0, scene="room", res=round(_log_uniform(rng, 0.015, 0.04), 4))
        if kind in ("online", "score"):
            case["frames"] = min(case["frames"], 4)
        passes = max(case["iters"], 1) * (case["frames"] / 2 if kind == "online" else 1)
        if _updates(case) < 1.2e9 and _updates(case) * passes < 1.2e10:
            return case


def _params(case, shape):
    p = gvdb_params()
    p.rows, p.cols = shape
    p.K = _intrinsics(case, shape)
    p.res, p.prior, p.dims = float(case["res"]), 0.1, np.asarray(DIMS[case["scene"]], np.float32)
    p.const_sigmasq_poly = [float(case.get("sigma", 1.5 * p.res)), 0.0, 0.0]
    p.acc_thresh = 0.1
    p.activation = _lib.ACT_FULL_RAY if case["activation"] == "full" else _lib.ACT_ENDPOINT
    p.brick_local_vis = _lib.VIS_BRICK_LOCAL if case["vis"] == "brick" else _lib.VIS_CARRY
    return p


def _intrinsics(case, shape):
    rows, cols = shape
    if not case["rows"]:
        return synth.intrinsics(rows, cols)
    f = case["focal"] * cols
    return np.array([[f, 0, (cols - 1) / 2], [0, f, (rows - 1) / 2], [0, 0, 1]], np.float32)


def _keyframes(case, seed):
    """(params, [(pose, K, depth)], scene): a scene of its own for each seed."""
    scene = synth.Scene(case["scene"], 1 + seed % 1000003)
    rng = np.random.default_rng(seed)
    n, frames = case["frames"], []
    for k in range(n):
        # the uneven keyframes go through the three cameras in turn
        shape = (case["rows"], case["cols"]) if case["rows"] else UNEVEN[k % len(UNEVEN)]
        K, pose = _intrinsics(case, shape), scene.ring_pose(k, n)
        frames.append((pose, K, scene.render(pose, K, *shape, noise_seed=int(rng.integers(1 << 40)))))
    return _params(case, frames[0][2].shape), frames, scene


def _context(params, frames):
    g = GVDBInference(params=params)
    for pose, K, depth in frames:
        g.add_camera_with_depth(pose, depth, K)
    return g


def _external_map(case, scene, seed):
    """Occupied leaves of an octree map of the scene: voxel centres and occupancies."""
    n = [int(round(d / case["res"])) for d in DIMS[case["scene"]]]
    vox = np.stack(np.meshgrid(*[np.arange(m, dtype=np.float32) for m in n], indexing="ij"), -1).reshape(-1, 3) + 0.5
    world = (vox - np.array([n[0] / 2, n[1] / 2, 0], np.float32)) * np.float32(case["res"])
    # the solid objects, and the walls as the outermost voxels of the room
    edge = ((vox < 1) | (vox > np.array(n, np.float32) - 1)).any(1)
    pts = vox[edge | (scene.occupancy(world) > 0)]
    occ = np.random.default_rng(seed).uniform(0.55, 0.97, len(pts)).astype(np.float32)
    return pts, occ


def _moved(pose):
    """A pose corrected by 2 cm and half a degree about the vertical."""
    c, s = math.cos(math.radians(0.5)), math.sin(math.radians(0.5))
    out = np.array(pose, np.float32)
    out[:3, :3] = (np.array([[c, -s, 0], [s, c, 0], [0, 0, 1]]) @ out[:3, :3]).astype(np.float32)
    out[0, 3] += 0.02
    return out


class _State:
    pass


def _grid_bricks(case):
    n = 1
    for d in DIMS[case["scene"]]:
        n *= (int(round(d / case["res"])) + 7) // 8
    return n


def prepare(case, seed):
    st = _State()
    st.case, st.kind = case, case["kind"]
    if st.kind == "train":
        st.X, st.t, st.w0 = _training_set(case, seed)
        st.g = GVDBInference(params=gvdb_params())
        return st
    st.params, st.frames, scene = _keyframes(case, seed)
    # readback buffers for the largest map the room can hold; a map fills its first rows
    st.bricks = np.zeros((_grid_bricks(case), 3), np.float32)
    st.alphas = np.zeros((_grid_bricks(case), 512), np.float32)
    if st.kind == "load":
        st.points, st.occ = _external_map(case, scene, seed)
    if st.kind in ("refine", "repose", "score"):
        st.g = _context(st.params, st.frames)
        if st.kind == "refine":
            st.g.prepare()
        else:
            st.g.perform_inference(max_iters=case["iters"])
        st.poses = [_moved(st.frames[0][0]), st.frames[0][0]]
        st.turn = 0
    return st


def _training_set(case, seed):
    """Features and targets as the warm start's samples have them: saturated
    free space and voxels near surfaces, 27 neighbour beliefs each."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    X = np.zeros((n, _lib.MLP_FEATURES), np.float32)
    near = rng.random(n) < 0.6
    X[:, 0] = np.where(near, np.log1p(rng.poisson(2.0, n)), 0)
    X[:, 1] = np.log1p(rng.gamma(2.0, 8.0, n))
    X[:, 2] = np.clip(rng.normal(-0.3, 0.25, n), -1, 1)
    X[:, 3] = np.clip(X[:, 2] + rng.exponential(0.2, n), -1, 1)
    X[:, 4] = np.where(near, np.sqrt(rng.integers(0, 16, n)) / 4, 1)
    X[:, 5:] = np.clip(X[:, 2:3] + rng.normal(0, 0.3, (n, 27)), -3, 3)
    t = np.clip(9.21 * (X[:, 3] + 0.3 * X[:, 0] - 0.8 * X[:, 4]) + rng.normal(0, 0.5, n), -9.21, 9.21)
    w0 = np.zeros(_lib.MLP_PARAMS, np.float32)
    for at, count, fan in ((0, 2048, 32), (2112, 4096, 64), (6272, 64, 64)):  # W1, W2, w3; biases 0
        w0[at:at + count] = rng.uniform(-1, 1, count) * math.sqrt(6 / fan)
    w0[-1] = -9.21
    return X, t.astype(np.float32), w0


def _read(st, g):
    n = g.num_bricks()
    st.bricks[:n] = g.get_occupied_bricks()
    g.get_indices_and_alphas(st.alphas[:n])
    return {"bricks": st.bricks, "alphas": st.alphas}


def run(state):
    st, kind = state, state.kind
    if kind == "refine":
        st.g.perform_inference(max_iters=st.case["iters"])
        return _read(st, st.g)
    if kind == "repose":
        st.g.set_pose(0, st.poses[st.turn])
        st.turn ^= 1
        st.g.perform_inference(max_iters=st.case["iters"])
        return _read(st, st.g)
    if kind == "score":
        return [st.g.evaluate(cam_id=k) for k in range(len(st.frames))]
    if kind == "train":
        w, losses = st.g.mlp_train(st.w0, st.X, st.t, epochs=st.case["epochs"], batch=st.case["batch"], lr=2e-3)
        return {"weights": w, "losses": losses}
    if kind == "load":
        g = GVDBMapLikelihoodEstimator(params=st.params)
        g.load_map(st.points, st.occ)
        pose, K, depth = st.frames[0]
        out = g.evaluate(pose=pose, depth=depth, K=K)
    else:
        g = GVDBInference(params=st.params)
        for k, (pose, K, depth) in enumerate(st.frames):
            g.add_camera_with_depth(pose, depth, K)
            if kind == "online":
                g.perform_inference(max_iters=st.case["iters"])
        if kind == "build":
            g.perform_inference(max_iters=st.case["iters"])
        out = _read(st, g)
    g.close()
    return out


def work(case):
    """Bytes and operations of one pass, whatever the code does."""
    kind = case["kind"]
    if kind == "train":
        # features and targets once per epoch; forward 2 x 6144 multiply-adds, backward twice that
        n = case["n"] * case["epochs"]
        return {"bytes": n * 33 * 4 + 2 * _lib.MLP_PARAMS * 4, "flops": n * 6 * 6144}
    vox = np.prod([d / case["res"] for d in DIMS[case["scene"]]])
    upd = _updates(case)
    if kind in ("load", "score"):
        # every ray crosses the whole room once: its voxels' beliefs and four images
        pix = case["frames"] * case["rows"] * case["cols"]
        return {"bytes": upd * 4 + pix * 20, "flops": upd * 40}
    # an incidence is a voxel index and a chord length (8 B) and a message (4 B) per iteration
    passes = case["iters"] * ((case["frames"] + 1) / 2 if kind == "online" else 1)
    build = {"refine": 0, "repose": 1 / case["frames"]}.get(kind, 1)
    return {"bytes": upd * (12 * passes + 8 * build) + vox * 4, "flops": upd * 50 * passes}


# ---------------------------------------------------------------- 64-bit outputs
class _Exact:
    """Traversal, BP and map scoring of full-ray maps in 64 bits, all rays of
    a keyframe at a time, step by step along the rays (dense voxel arrays)."""

    def __init__(self, p):
        self.p, self.dev = p, "cuda" if torch.cuda.is_available() else "cpu"
        m = [int(round(float(d) / float(p.res))) for d in p.dims]
        self.N = [(v + 7) // 8 * 8 for v in m]
        self.off = [0.5 * m[0], 0.5 * m[1], 0.0]
        self.nvox = self.N[0] * self.N[1] * self.N[2]
        self.res = float(np.float32(p.res))
        self.sigma = float(np.float32(p.const_sigmasq_poly[0]))  # constant, and no bias
        self.brick = p.brick_local_vis == _lib.VIS_BRICK_LOCAL

    def full(self, n, v=0.0, dtype=torch.float64):
        return torch.full((n,), v, dtype=dtype, device=self.dev)

    def rays(self, pose, K, shape):
        """Fixed-point origins and directions (voxels, 2^-16), |D| per metre."""
        pose, K = np.asarray(pose, np.float64), np.asarray(K, np.float64)
        y, x = np.mgrid[0:shape[0], 0:shape[1]].reshape(2, -1)
        u = np.stack([(x - K[0, 2]) / K[0, 0], (y - K[1, 2]) / K[1, 1], np.ones(x.size)])
        Di = np.rint(pose[:3, :3] @ u / self.res * 65536)
        Oi = np.rint((pose[:3, 3] / self.res + self.off) * 65536)
        norm = np.sqrt(((Di / 65536) ** 2).sum(0))
        to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)  # noqa: E731
        return Oi, to(Di), to(norm)

    def walk(self, pose, K, shape, depth=None):
        """Steps of every ray through the map: per step the rays still going,
        their voxel, chord length, entry and exit depth, whether the voxel
        starts a brick and whether the walk leaves a brick after it.  With
        depth, a ray ends at the first brick exit past d + 3 sigma."""
        Oi, Di, norm = self.rays(pose, K, shape)
        on = torch.ones(Di.shape[1], dtype=torch.bool, device=self.dev) if depth is None else depth > 0
        top = torch.tensor(self.N, dtype=torch.float64, device=self.dev)[:, None]
        inf = torch.tensor(math.inf, dtype=torch.float64, device=self.dev)
        O = torch.tensor(Oi, device=self.dev)[:, None]
        # entry into the grid (0 from inside it) and exit; rays that miss it are left out
        lo = torch.where(Di > 0, -O / Di, (top * 65536 - O) / Di)
        hi = torch.where(Di > 0, (top * 65536 - O) / Di, -O / Di)
        aside = (Di == 0) & ((O < 0) | (O >= top * 65536))
        lo, hi = torch.where(Di == 0, -inf, lo), torch.where(Di == 0, inf, hi)
        zin, axis = lo.max(0)
        inside = zin <= 0
        zin = zin.clamp_min(0)
        ids = torch.nonzero(on & (zin < hi.min(0).values) & ~aside.any(0)).flatten()
        Di, norm, z0, axis, inside = Di[:, ids], norm[ids], zin[ids], axis[ids], inside[ids]
        d = None if depth is None else depth[ids]
        # the voxel there: floor of (O + zin D) / 2^16, exact in integers, the one below on a face met downwards
        Ea, Da = O.expand_as(Di).gather(0, axis[None])[0], Di.gather(0, axis[None])[0]
        face = torch.where(Da > 0, 0.0, top.flatten()[axis] * 65536)
        num = torch.where(inside, 0.0, (face - Ea) * torch.sign(Da)).long()
        den = torch.where(inside, 1.0, Da.abs()).long()
        X = O.long() * den + num * Di.long()
        sg = torch.sign(Di)
        ix = torch.div(X, den * 65536, rounding_mode="floor") - ((sg < 0) & (X % (den * 65536) == 0)).long()
        ix = ix.double().clamp_min(0).minimum(top - 1)
        first = torch.ones_like(norm, dtype=torch.bool)
        steps, ran_out = [], torch.zeros(on.numel(), dtype=torch.bool, device=self.dev)
        while ids.numel():
            t = torch.where(sg == 0, inf, ((ix + (sg > 0).double()) * 65536 - O) / Di)
            z1 = t.min(0).values
            nx = ix + sg * (t == z1).double()  # every tied axis steps
            vox = ((ix[0] * self.N[1] + ix[1]) * self.N[2] + ix[2]).long()
            length = ((z1 - z0) * norm).float().double()
            if int(vox.min()) < 0 or int(vox.max()) >= self.nvox:
                raise ValueError("a ray outside the grid")
            out = ((nx < 0) | (nx >= top)).any(0)
            end = out | (torch.floor(nx / 8) != torch.floor(ix / 8)).any(0)
            steps.append((ids, vox, length, z0, z1, first, end, ix))
            stop = out.clone()
            if d is not None:
                past = end & (z1 >= d + 3 * self.sigma)
                ran_out[ids[out & ~past & (d > z1)]] = True
                stop |= past
            keep = ~stop
            ids, Di, norm, sg, ix = ids[keep], Di[:, keep], norm[keep], sg[:, keep], nx[:, keep]
            z0, first = z1[keep], end[keep]
            d = None if d is None else d[keep]
        return steps, ran_out

    # -- BP
    def start(self):
        self.B = self.full(self.nvox, math.log(self.p.prior) - math.log1p(-self.p.prior))
        self.upd = self.full(self.nvox, False, torch.bool)
        self.cams, self.bricks = [], []

    def add(self, pose, K, depth):
        d = torch.from_numpy(depth.astype(np.float64).ravel()).to(self.dev)
        steps, ran_out = self.walk(pose, K, depth.shape, d)
        seen = self.full(self.nvox // 512, False, torch.bool)
        recs = []
        for ids, vox, length, _, z1, first, _, ix in steps:
            b = torch.floor(ix / 8).long()
            seen[(b[0] * (self.N[1] // 8) + b[1]) * (self.N[2] // 8) + b[2]] = True
            u = (d[ids] - z1).abs() / (3 * self.sigma)
            recs.append((ids, vox, length, 0.398942 * torch.exp(-u * u / 2), first))
        # sums per voxel over the rays, in record order: a sort once, then segments
        sums = (None, None, None)
        if recs:
            vox, order = torch.sort(torch.cat([r[1] for r in recs]), stable=True)
            sums = (*torch.unique_consecutive(vox, return_counts=True), order)
        C = self.per_voxel(sums, [r[2] for r in recs])
        self.cams.append((recs, ran_out, C, self.full(self.nvox), d.numel(), sums))
        return seen

    def per_voxel(self, sums, values):
        out = self.full(self.nvox)
        if values:
            voxels, counts, order = sums
            out[voxels] = torch.segment_reduce(torch.cat(values)[order], "sum", lengths=counts)
        return out

    def infer(self, iters):
        for cam in self.cams:
            cam[3].zero_()  # a call starts from empty messages
        for _ in range(iters):
            for cam in self.cams:
                self.camera_pass(*cam)

    def camera_pass(self, recs, ran_out, C, M, nrays, sums):
        n = (1 / (1 + torch.exp(self.B - M))).clamp(F_EPS, 1 - F_EPS)
        tiny = 2.0 ** -126
        T, L, nz = self.full(nrays), self.full(nrays), self.full(nrays, False, torch.bool)
        for ids, vox, length, a, first in recs:
            nn, Lr = n[vox], L[ids]
            psi = a / (3 * self.sigma)
            if self.brick:  # visibility starts again at each brick until a tau survives 32-bit flushing
                Lr = torch.where(first & ~nz[ids], torch.zeros_like(Lr), Lr)
            Lr = Lr + length * torch.log(nn)
            b = torch.exp(Lr) * (1 - nn)
            tau = b * psi
            if self.brick:
                counts = torch.minimum(torch.minimum(a, psi), torch.minimum(b, tau)) >= tiny
                nz[ids] |= counts
                tau = torch.where(counts, tau, torch.zeros_like(tau))
            T[ids] += tau
            L[ids] = Lr
        T = T + torch.where(ran_out, torch.exp(L), torch.zeros_like(L))
        P, L, sent = self.full(nrays), self.full(nrays), []
        for ids, vox, length, a, _ in recs:
            nn, Pr = n[vox], P[ids]
            Lr = L[ids] + length * torch.log(nn)
            vpsi = torch.exp(Lr) * a / (3 * self.sigma)
            tau = vpsi * (1 - nn)
            mu1 = Pr + vpsi
            mu0 = Pr + (T[ids] - Pr - tau) / nn
            sent.append((mu1 / (mu1 + mu0 + 1e-7)).clamp(F_EPS, 1 - F_EPS) * length)
            P[ids], L[ids] = Pr + tau, Lr
        S = self.per_voxel(sums, sent)
        on = C > float(np.float32(0.1))
        q = (S / torch.where(on, C, torch.ones_like(C))).clamp(F_EPS, 1 - F_EPS)
        m = torch.log(q) - torch.log1p(-q)
        self.B = torch.where(on, self.B + m - M, self.B)
        M.copy_(torch.where(on, m, M))
        self.upd |= on

    def grow(self, seen):
        """Bricks join in ascending order, after those already there."""
        known = set(self.bricks)
        self.bricks += [b for b in torch.nonzero(seen).flatten().tolist() if b not in known]

    def map(self):
        nb = [v // 8 for v in self.N]
        lin = np.asarray(self.bricks)
        xyz = np.stack([lin // (nb[1] * nb[2]), lin // nb[2] % nb[1], lin % nb[2]], 1) * 8
        alpha = 1 - (1 / (1 + torch.exp(self.B))).clamp(F_EPS, 1 - F_EPS)
        grid = torch.where(self.upd, alpha, torch.zeros_like(alpha)).reshape(self.N).cpu().numpy()
        bricks, rows = np.zeros((self.nvox // 512, 3)), np.zeros((self.nvox // 512, 512))
        for k, (x, y, z) in enumerate(xyz):
            bricks[k] = x + 4, y + 4, z + 4
            rows[k] = grid[x:x + 8, y:y + 8, z:z + 8].ravel()
        return {"bricks": bricks, "alphas": rows}

    # -- scoring of a loaded map
    def load(self, pts, occ):
        v = np.floor(pts.astype(np.float64)).astype(np.int64)
        lin = (v[:, 0] * self.N[1] + v[:, 1]) * self.N[2] + v[:, 2]
        alpha, active = np.zeros(self.nvox), np.zeros([n // 8 for n in self.N], bool)
        alpha[lin] = np.clip(occ.astype(np.float64), F_EPS, 1 - F_EPS)
        lo, hi = np.maximum(v - 1, 0) // 8, np.minimum(v + 1, np.array(self.N) - 1) // 8
        for c in range(8):  # bricks within a voxel of a point
            b = np.where([c & 1, c >> 1 & 1, c >> 2 & 1], hi, lo)
            active[b[:, 0], b[:, 1], b[:, 2]] = True
        self.alpha, self.active = (torch.from_numpy(a).to(self.dev) for a in (alpha, active))

    def score(self, pose, K, depth):
        d = torch.from_numpy(depth.astype(np.float64).ravel()).to(self.dev)
        steps, _ = self.walk(pose, K, depth.shape)
        vis, total, esum = self.full(d.numel(), 1.0), self.full(d.numel()), self.full(d.numel())
        lam, before, started = self.full(d.numel()), self.full(d.numel()), self.full(d.numel(), False, torch.bool)
        axis, t = np.asarray(pose, np.float64)[:3, 2], np.asarray(pose, np.float64)[:3, 3]
        psi = lambda s, dd: 0.398942 * torch.exp(-0.5 * ((dd - s) / (3 * self.sigma)) ** 2) / (3 * self.sigma)  # noqa: E731
        for ids, vox, length, z0, z1, _, _, ix in steps:
            b = torch.floor(ix / 8).long()
            on = self.active[b[0], b[1], b[2]]
            ids, vox, length, z0, z1, ix = ids[on], vox[on], length[on], z0[on], z1[on], ix[:, on]
            s0 = torch.where(started[ids], before[ids], z0)
            lam[ids] += torch.log1p(-self.alpha[vox]) * length
            v1 = torch.exp(lam[ids])
            w = vis[ids] - v1
            dd = d[ids]
            near = (z1 - dd).abs() <= 3 * self.sigma
            prob = torch.where(near, 0.999 * 0.5 * (psi(z1, dd) + psi(s0, dd)), torch.full_like(dd, 1e-3))
            total[ids] += w * torch.where(z1 < 0.1, torch.zeros_like(prob), prob)
            zc = sum(axis[a] * ((ix[a] + 0.5 - self.off[a]) * self.res - t[a]) for a in range(3))
            esum[ids] += w * zc
            vis[ids], before[ids], started[ids] = v1, z1, True
        ll = torch.log(total + vis * torch.where(d >= 10, 0.999, 1e-3))
        ll = torch.where(d > 0, ll, torch.zeros_like(ll))
        depth_image = esum / (1 - vis + F_EPS)
        return {"loglik": ll.reshape(depth.shape).cpu().numpy(), "log_likelihood": float(ll.sum()),
                "expected_depth": depth_image.reshape(depth.shape).cpu().numpy()}


def exact(case, seed):
    """64-bit outputs, where they take seconds: small full-ray maps and loaded
    maps.  The class images and counts are decisions, not computed numbers."""
    kind = case["kind"]
    if kind == "load":
        params, frames, scene = _keyframes(case, seed)
        e = _Exact(params)
        e.load(*_external_map(case, scene, seed))
        none = dict.fromkeys(("accuracy", "simple_accuracy", "accuracy_counts", "simple_counts", "accuracy_image",
                              "simple_accuracy_image"))
        pose, K, depth = frames[0]
        return dict(none, **e.score(pose, K, depth))
    if kind not in ("build", "refine", "online") or case["activation"] != "full" or not case["rows"]:
        return None
    passes = case["iters"] * case["frames"] * ((case["frames"] + 1) / 2 if kind == "online" else 1)
    steps = 1.3 * sum(DIMS[case["scene"]]) / case["res"]
    if passes * steps > 60000 or case["frames"] * case["rows"] * case["cols"] * steps > 8e8:
        return None
    params, frames, _ = _keyframes(case, seed)
    e = _Exact(params)
    e.start()
    seen = []
    for pose, K, depth in frames:
        seen.append(e.add(pose, K, depth))
        if kind == "online":
            e.grow(seen[-1])
            e.infer(case["iters"])
    if kind != "online":
        e.grow(torch.stack(seen).any(0))
        e.infer(case["iters"])
    return e.map()
