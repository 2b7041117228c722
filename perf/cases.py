"""What is timed of this framework: the calls that its users make, over the sizes they make them at.

A case is a dict of plain values.  `kind` says which part of the framework it goes through:

  cycles     a context stepped as the server's runner does it: one cycle, one frame of renderable
             positions, cycle after cycle, and the body state read back at the end
  surrogate  the same with the learned far field, its network trained beforehand on other scenes
  octree     the same with the Barnes-Hut octree
  batch      many small simulations advanced together
  churn      the collection's bookkeeping: a delete request, queued adds, Cycle, one frame
  training   the far field's network trained on rows that the caller holds

State outputs are the FP64 body state; frames are FP32.  Every pass continues from the state that
the last one left, as a program's next call does.
"""
import math

import numpy as np
import torch

from nbodygo_amd import Bodies, NBodyBatch, NBodyGPU, gen
from nbodygo_amd import _lib as L
from nbodygo_amd.mlp import MLP

DT = 1e-3        # the runner's time scaling in the benchmark and the tests
SOFT = 0.01      # Plummer softening of the benchmark's spheres


def listed():
    return [
        # The server's default scene: 1,000 bodies, the reference's gravity and elastic collisions
        # in FP64.  The smallest calls: what a cycle costs beside its arithmetic.
        dict(name="server_fp64_1k", kind="cycles", n=1000, scene="uniform", precision="fp64",
             collisions=True, radius=0.05, cycles=10),
        # The same scene grown to a ragged size on the FP32 production path (exact overlap gate,
        # no softening): an interactive session with many bodies.
        dict(name="server_fp32_10k", kind="cycles", n=10007, scene="uniform", precision="fp32",
             collisions=True, radius=0.05, cycles=10),
        # FP64 in the reference's operation order at a size where arithmetic counts: validation
        # runs against the Go server.
        dict(name="fp64_16k", kind="cycles", n=16384, scene="uniform", precision="fp64",
             collisions=True, radius=0.05, cycles=2),
        # A Plummer sphere with elastic collisions, the ordinary direct-sum run.
        dict(name="elastic_65k", kind="cycles", n=65536, scene="plummer", precision="fp32",
             collisions=True, radius=1e-4, cycles=2),
        # The headline: a large direct sum without collisions.
        dict(name="plain_262k", kind="cycles", n=262144, scene="plummer", precision="fp32",
             collisions=False, radius=0.0, cycles=2),
        # A parameter sweep: 512 Plummer spheres of 256 to 8,192 bodies.
        dict(name="batch_512", kind="batch", sims=512, lo=256, hi=8192, sizes=7, cycles=4),
        # The headline sphere with the learned far field, its error checked at every step.
        dict(name="surrogate_262k", kind="surrogate", n=262144, scene="plummer", collisions=False,
             grid=32, shell=2, train_sims=3, train_rows=2048, fit_steps=600, tol=1e-3, cycles=5),
        # Two colliding spheres with collisions and the learned far field: the largest scene.
        dict(name="collide_1m", kind="surrogate", n=1048576, scene="two", collisions=True,
             grid=64, shell=3, train_sims=1, train_rows=4096, fit_steps=600, tol=5e-3, cycles=4),
        # The reference's own far-field design in its FP64 arithmetic, a ragged size.
        dict(name="octree_exact_100k", kind="octree", n=100003, mode="exact", theta=0.3, cycles=2),
        # The octree's fast mode at the headline's size.
        dict(name="octree_fast_262k", kind="octree", n=262144, mode="fast", theta=0.3, cycles=4),
        # A server that deletes and adds 1 % of a million bodies in one cycle.
        dict(name="churn_1m", kind="churn", n=1048576, remove=10485, add=10485),
        # The far field's network: forward, backward and the optimiser.
        dict(name="training", kind="training", rows=8192, batch=512, steps=200),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fp64", "fp32", "fp32", "plain", "batch", "surrogate", "octree", "octree",
                       "churn", "training"])
    if kind == "fp64":
        return dict(kind="cycles", n=_log_int(rng, 200, 20000), scene="uniform", precision="fp64",
                    collisions=rng.random() < 0.75, radius=0.05, cycles=2)
    if kind == "fp32":
        if rng.random() < 0.5:
            return dict(kind="cycles", n=_log_int(rng, 500, 60000), scene="uniform",
                        precision="fp32", collisions=rng.random() < 0.75, radius=0.05, cycles=2)
        return dict(kind="cycles", n=_log_int(rng, 1000, 100000), scene="plummer",
                    precision="fp32", collisions=True, radius=10 ** rng.uniform(-4.5, -3.0),
                    cycles=1)
    if kind == "plain":
        return dict(kind="cycles", n=_log_int(rng, 2000, 262144), scene="plummer",
                    precision="fp32", collisions=False, radius=0.0, cycles=1)
    if kind == "batch":
        lo = _log_int(rng, 64, 1024)
        return dict(kind="batch", sims=_log_int(rng, 8, 512), lo=lo,
                    hi=_log_int(rng, 2 * lo, 8192), sizes=rng.randrange(1000), cycles=2)
    if kind == "surrogate":
        return dict(kind="surrogate", n=_log_int(rng, 30000, 262144), scene="plummer",
                    collisions=rng.random() < 0.3, grid=32, shell=rng.choice([2, 2, 3]),
                    train_sims=2, train_rows=2048, fit_steps=400, tol=5e-3, cycles=3)
    if kind == "octree":
        return dict(kind="octree", n=_log_int(rng, 5000, 200000),
                    mode=rng.choice(["exact", "fast"]), theta=rng.choice([0.3, 0.3, 0.5]),
                    cycles=2)
    if kind == "churn":
        n = _log_int(rng, 10000, 1048576)
        k = max(1, int(n * rng.uniform(0.001, 0.02)))
        return dict(kind="churn", n=n, remove=k, add=k)
    batch = rng.choice([128, 256, 512, 1024])
    return dict(kind="training", rows=batch * rng.randrange(4, 17), batch=batch,
                steps=rng.randrange(50, 200))


def _scene(case, seed):
    n = case["n"]
    if case["scene"] == "uniform":
        return gen.uniform_sphere(n, seed, radius_k=case["radius"])
    if case["scene"] == "two":
        return gen.two_plummer(n // 2, seed, radius_k=0.05 if case["collisions"] else 0.0)
    if case["kind"] == "surrogate" and case["collisions"]:
        return gen.plummer(n, seed, radius=1e-4)
    return gen.plummer(n, seed, radius=case.get("radius", 0.0))


def _network(case, seed):
    """Rows and weights as the far field has them: 30 features of order one, 3 residuals, weights
    of the usual initial size."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["rows"], 30), dtype=np.float32)
    mix = rng.standard_normal((30, 3)).astype(np.float32) / np.float32(30 ** 0.5)
    t = np.tanh(x @ mix).astype(np.float32)
    parts, dims = [], [30, 128, 128, 128, 3]
    for i, o in zip(dims[:-1], dims[1:]):
        parts += [(rng.standard_normal(i * o) / i ** 0.5).astype(np.float32),
                  np.zeros(o, np.float32)]
    return x, t, np.concatenate(parts)


def _clusters(case, seed):
    sizes = gen.batch_sizes(case["sims"], case["sizes"], case["lo"], case["hi"])
    return [gen.plummer(int(n), seed * 100003 + k) for k, n in enumerate(sizes)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return dict(case=case, g=NBodyBatch(G=1.0, eps=SOFT).load(_clusters(case, seed)))
    if kind == "training":
        x, t, p = _network(case, seed)
        net = MLP(30, hidden=128, layers=3, d_out=3, seed=1)
        net.set_params(p)
        return dict(case=case, g=net, x=x, t=t)
    if kind == "churn":
        g = NBodyGPU(G=1.0, eps=SOFT, overlap_cutoff=False, collisions=False)
        g.load(gen.plummer(case["n"], seed))
        return dict(case=case, g=g, add=gen.plummer(case["add"], seed + 1000))
    if kind == "octree":
        g = NBodyGPU(G=1.0, eps=0.0, overlap_cutoff=False, collisions=False, precision="fp64")
        g.load(gen.plummer(case["n"], seed))
        g.bh_enable(theta=case["theta"], mode=case["mode"])
        return dict(case=case, g=g)
    if kind == "surrogate":
        g = NBodyGPU(G=1.0, eps=SOFT, overlap_cutoff=False, collisions=case["collisions"])
        opts = dict(grid=case["grid"], shell=case["shell"])
        for k in range(case["train_sims"]):
            g.load(_scene(case, seed + 1000 + 2 * k))
            g.sur_enable(check_every=0, **opts)
            g.sur_collect(case["train_rows"], seed=k)
        g.sur_fit(steps=case["fit_steps"], batch=512, lr=1e-3)
        g.load(_scene(case, seed))
        g.sur_enable(check_every=1, tol=case["tol"], **opts)
        return dict(case=case, g=g)
    if case["scene"] == "uniform":  # the reference's force: its G, no softening, the overlap gate
        g = NBodyGPU(collisions=case["collisions"], precision=case["precision"])
    else:
        g = NBodyGPU(G=1.0, eps=SOFT, overlap_cutoff=False, collisions=case["collisions"],
                     precision=case["precision"])
    g.load(_scene(case, seed))
    return dict(case=case, g=g)


def _state(b: Bodies):
    return dict(pos=[b.x, b.y, b.z], vel=[b.vx, b.vy, b.vz], flags=b.flags)


def run(state):
    case, g = state["case"], state["g"]
    kind = case["kind"]
    if kind == "batch":
        g.step(DT, 1.0, nsteps=case["cycles"])
        return _state(g.store())
    if kind == "training":
        loss = g.train(state["x"], state["t"], steps=case["steps"], batch=case["batch"], lr=1e-3)
        return dict(weights=g.get_params(), loss=np.float32(loss))
    if kind == "churn":
        removed = g.remove_bodies(case["remove"])
        g.add_bodies(state["add"])
        n = g.cycle(1.0)
        xyz, exists = g.render()
        return dict(removed=removed, n=n, frame=xyz, exists=exists)
    pairs = 0
    for _ in range(case["cycles"]):
        pairs += g.step(DT, 1.0)["pairs_total"]
        xyz, exists = g.render()
    return dict(frame=xyz, exists=exists, pairs=pairs, **_state(g.store()))


def work(case):
    """Bytes: the state read and written once, the frames written.  Operations: a direct sum takes
    26 for each unordered pair (differences 3, squared distance 6, reciprocal square root and its
    cube 3, two masses, two three-component accumulations 12); the far fields take at least 60
    terms of 20 operations a body; training 6 per weight and row."""
    kind = case["kind"]
    if kind == "training":
        weights = 30 * 128 + 2 * 128 * 128 + 128 * 3
        return dict(bytes=4.0 * (case["rows"] * 33 + 2 * weights),
                    flops=6.0 * weights * case["batch"] * case["steps"])
    if kind == "churn":
        return dict(bytes=2.0 * 93 * case["n"] + 13.0 * case["n"], flops=3.0 * case["n"])
    if kind == "batch":
        lo, hi, k = case["lo"], case["hi"], case["sims"]
        n, n2 = k * (lo + hi) / 2, k * (hi * hi + hi * lo + lo * lo) / 3
        return dict(bytes=97.0 * n * case["cycles"], flops=13.0 * n2 * case["cycles"])
    n, c = case["n"], case["cycles"]
    moved = (2.0 * 48 + 8 + 13) * n * c + 93.0 * n
    if kind in ("surrogate", "octree"):
        return dict(bytes=moved, flops=1200.0 * n * c)
    return dict(bytes=moved, flops=13.0 * n * (n - 1) * c)


def _accel64(x, m, eps2, chunk):
    a = torch.empty_like(x)
    for i in range(0, x.shape[0], chunk):
        d = x[None, :, :] - x[i:i + chunk, None, :]
        r2 = d.square().sum(-1).add_(eps2)
        w = r2.rsqrt_().pow_(3).mul_(m)
        a[i:i + chunk] = (w[..., None] * d).sum(1)
    return a


def _cycles64(parts, cycles):
    """Softened direct sum (G = 1) and semi-implicit Euler on each part, in 64 bits."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pos, vel = [], []
    for b in parts:
        x, v = (torch.from_numpy(q).to(dev) for q in (b.pos(), b.vel()))
        m = torch.from_numpy(b.m).to(dev)
        for _ in range(cycles):
            v = v + DT * _accel64(x, m, SOFT * SOFT, max(1, (1 << 26) // b.n))
            x = x + DT * v
        pos.append(x.cpu().numpy())
        vel.append(v.cpu().numpy())
    return np.concatenate(pos), np.concatenate(vel)


def _network64(case, seed):
    """The training loop in 64 bits: mean squared error over consecutive minibatches, Adam."""
    x, t, p = _network(case, seed)
    x, t = torch.from_numpy(x).double(), torch.from_numpy(t).double()
    flat = torch.from_numpy(p).double().requires_grad_(True)
    opt = torch.optim.Adam([flat], lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    dims = [30, 128, 128, 128, 3]
    at = 0
    for _ in range(case["steps"]):
        if at + case["batch"] > case["rows"]:
            at = 0
        h, off = x[at:at + case["batch"]], 0
        for k, (i, o) in enumerate(zip(dims[:-1], dims[1:])):
            h = h @ flat[off:off + i * o].view(i, o) + flat[off + i * o:off + i * o + o]
            off += i * o + o
            if k < 3:
                h = torch.nn.functional.gelu(h, approximate="tanh")
        loss = (h - t[at:at + case["batch"]]).square().mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        at += case["batch"]
    return dict(weights=flat.detach().float().numpy().astype(np.float64), loss=None)


def exact(case, seed):
    """64-bit values where plain torch gives them: training, and the direct sums that no collision
    and no overlap gate bends.  The octree's value is defined by its tree, collisions by the
    reference's resolution: neither has a plain form."""
    kind = case["kind"]
    if kind == "training":
        return _network64(case, seed)
    if kind == "batch":
        pos, vel = _cycles64(_clusters(case, seed), case["cycles"])
        return dict(pos=list(pos.T.copy()), vel=list(vel.T.copy()), flags=None)
    if kind in ("cycles", "surrogate") and case["scene"] == "plummer" and not case["collisions"] \
            and case["n"] ** 2 * case["cycles"] < 1.6e11:
        pos, vel = _cycles64([_scene(case, seed)], case["cycles"])
        return dict(frame=pos, exists=None, pairs=None, pos=list(pos.T.copy()),
                    vel=list(vel.T.copy()), flags=None)
    return None
