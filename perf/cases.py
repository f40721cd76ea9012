"""The calls that users of this framework make, as timed cases.

QuickSampling realisations (`g2s_amd.qs`) are the main work: a training image
and a grid to simulate go in as host arrays, the simulated grid and the index
image come back, so a pass is the whole call. Beside them stand the calls of
a program that drives its own path (one node at a time, or a wave of nodes at
once), the parameter calibration, and the gradient of the learned proposal.

Training images are Gaussian random fields with an exponential covariance
(periodic spectral synthesis), passed through exp() or thresholded into
classes as the benchmark's are. Everything follows from the seed.
"""
import math

import numpy as np
import torch

import g2s_amd
from g2s_amd import lp as g2s_lp

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
# x, y, z: training image (z = 0: 2-D); sx, sy, sz: simulated grid; n
# neighbours; k best; hard: share of the simulated cells that are given.
_LISTED = [
    # first look at a small image: the whole call is launches and set-up
    dict(name="qs_small", family="qs", kind="cont", x=80, y=64, z=0, sx=24, sy=20, sz=0, n=12, k=1.5, classes=0,
         hard=0.0),
    # binary facies, the full 200 x 200 realisation of the 2-D categorical workload
    dict(name="qs_cat_2d", family="qs", kind="cat", x=250, y=250, z=0, sx=200, sy=200, sz=0, n=50, k=1.2, classes=2,
         hard=0.0),
    # continuous 2-D image of ordinary, ragged size with conditioning data
    dict(name="qs_cont_2d", family="qs", kind="cont", x=271, y=233, z=0, sx=120, sy=150, sz=0, n=40, k=1.5, classes=0,
         hard=0.05),
    # the benchmark's image and parameters on a part of its grid
    dict(name="qs_cont_2d_large", family="qs", kind="cont", x=1000, y=1000, z=0, sx=220, sy=220, sz=0, n=80, k=1.5,
         classes=0, hard=0.0),
    # co-located continuous and 4-class variables, 10 % hard data
    dict(name="qs_multi_2d", family="qs", kind="multi", x=500, y=500, z=0, sx=160, sy=160, sz=0, n=60, k=1.5,
         classes=4, hard=0.1),
    # three facies in 3-D, the image and parameters of the 3-D workload
    dict(name="qs_cat_3d", family="qs", kind="cat", x=180, y=150, z=120, sx=24, sy=24, sz=12, n=100, k=1.5, classes=3,
         hard=0.0),
    # a continuous property in 3-D (porosity, permeability) with well data
    dict(name="qs_cont_3d", family="qs", kind="cont", x=100, y=90, z=50, sx=22, sy=20, sz=12, n=30, k=1.5, classes=0,
         hard=0.03),
    # a host program's own path loop hands over 256 nodes at once
    dict(name="wave_256", family="wave", x=1000, y=1000, nodes=256, n=80, k=1.5),
    # the same loop one node at a time, as G2S's device interface is driven
    dict(name="node", family="node", x=400, y=300, nodes=1, n=40, k=1.5),
    # calibration with its default neighbour counts and densities
    dict(name="calibration", family="calib", x=1000, y=1000, kernel=201, max_nb=80, iters=2),
    # loss and gradient of one training batch of the learned proposal
    dict(name="proposal_gradient", family="grad", batch=256, keys=1024),
]


def listed():
    return [dict(c) for c in _LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    k = rng.choice((1.0, 1.2, 1.5, 2.0))
    if pick < 0.62:
        kind = rng.choice(("cont", "cont", "cat", "multi"))
        classes = {"cont": 0, "cat": rng.randint(2, 5), "multi": rng.randint(2, 4)}[kind]
        if rng.random() < 0.65:
            x, y = _log(rng, 70, 1000), _log(rng, 70, 1000)
            cells = _log(rng, 500, 40000)
            sx = max(16, min(250, int(math.sqrt(cells) * rng.uniform(0.7, 1.4))))
            sy = max(16, min(250, cells // sx))
            return dict(family="qs", kind=kind, x=x, y=y, z=0, sx=sx, sy=sy, sz=0, n=rng.randint(8, 90), k=k,
                        classes=classes, hard=rng.choice((0.0, 0.0, 0.05, 0.1)))
        kind = "cat" if kind == "multi" else kind
        classes = classes if kind == "cat" else 0
        x, y, z = _log(rng, 40, 180), _log(rng, 40, 150), _log(rng, 24, 120)
        cells = min(_log(rng, 800, 7000), int(2.0e10 / (x * y * z)))
        sz = rng.randint(5, 12)
        sx = max(8, min(30, int(math.sqrt(cells / sz) * rng.uniform(0.8, 1.2))))
        sy = max(8, min(30, cells // (sx * sz)))
        return dict(family="qs", kind=kind, x=x, y=y, z=z, sx=sx, sy=sy, sz=sz, n=rng.randint(10, 100), k=k,
                    classes=classes if kind == "cat" else 0, hard=rng.choice((0.0, 0.0, 0.03)))
    if pick < 0.76:
        return dict(family="wave", x=_log(rng, 100, 1000), y=_log(rng, 100, 1000), nodes=rng.randint(16, 256),
                    n=rng.randint(10, 80), k=k)
    if pick < 0.88:
        return dict(family="node", x=_log(rng, 60, 1000), y=_log(rng, 60, 1000), nodes=1, n=rng.randint(5, 80), k=k)
    if pick < 0.95:
        return dict(family="calib", x=_log(rng, 200, 1000), y=_log(rng, 200, 1000), kernel=2 * rng.randint(20, 100) + 1,
                    max_nb=rng.randint(20, 80), iters=1)
    return dict(family="grad", batch=rng.randint(32, 256), keys=rng.randint(512, 1024))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _field(shape, length, rng):
    """Standardised periodic Gaussian field (C order), exponential covariance."""
    lag = []
    for i, s in enumerate(shape):
        d = np.minimum(np.arange(s), s - np.arange(s)) / length[i]
        lag.append(torch.from_numpy((d ** 2).reshape([-1 if j == i else 1 for j in range(len(shape))])))
    h = sum(lag)
    lam = torch.fft.rfftn(torch.exp(-torch.sqrt(h))).real.clamp_min(0.0)
    white = torch.from_numpy(rng.standard_normal(shape))
    f = torch.fft.irfftn(torch.fft.rfftn(white) * torch.sqrt(lam), s=shape).numpy()
    return (f - f.mean()) / f.std()


def _lengths(shape):
    """Correlation lengths: 20 cells of a 1000-cell axis and 15 of a 250-cell
    one in 2-D, 25 / 25 / 6 of the 3-D workload's axes, shorter in small images."""
    if len(shape) == 3:
        return tuple(max(2.0, s / r) for s, r in zip(shape, (20.0, 6.0, 7.2)))
    return tuple(max(3.0, min(20.0, s / 16.0)) for s in shape)


def _image(kind, shape, classes, rng):
    """Values (cells, variables), dimension 0 fastest."""
    length = _lengths(shape)
    out = []
    if kind in ("cont", "multi"):
        a = _field(shape, length, rng)
        out.append(np.exp(a) if kind == "cont" else a)
    if kind in ("cat", "multi"):
        b = _field(shape, length, rng)
        if kind == "multi":
            b = 0.7 * out[0] + math.sqrt(1.0 - 0.49) * b
        edges = np.quantile(b, [0.72] if classes == 2 else np.arange(1, classes) / classes)
        out.append(np.digitize(b, edges))
    return np.stack([o.reshape(-1) for o in out], 1).astype(np.float32)


def _dims(c, a="x", b="y", d="z"):
    return (c[a], c[b]) + ((c[d],) if c[d] else ())


def _prepare_qs(c, seed):
    rng = np.random.default_rng([seed, 11])
    ti_dims, sim_dims = _dims(c), _dims(c, "sx", "sy", "sz")
    ti = _image(c["kind"], ti_dims[::-1], c["classes"], rng)
    di = np.full((int(np.prod(sim_dims)), ti.shape[1]), np.nan, np.float32)
    if c["hard"] > 0.0:
        given = rng.choice(di.shape[0], int(di.shape[0] * c["hard"]), replace=False)
        di[given] = _image(c["kind"], sim_dims[::-1], c["classes"], rng)[given]
    types = {"cont": [0], "cat": [1], "multi": [0, 1]}[c["kind"]]
    return dict(ti=ti, ti_dims=ti_dims, di=di, sim_dims=sim_dims, types=types, n=c["n"], k=c["k"], seed=seed)


def _offsets_by_distance(radius):
    a = np.arange(-radius, radius + 1)
    o = np.stack(np.meshgrid(a, a, indexing="ij"), -1).reshape(-1, 2)
    return o[np.argsort((o ** 2).sum(1), kind="stable")].astype(np.int32)


def _path_nodes(c, seed):
    """A continuous image and nodes as a path meets them: the node's own cell
    (no value), then the n nearest informed cells at some density."""
    rng = np.random.default_rng([seed, 12])
    shape = (c["y"], c["x"])
    ti = _image("cont", shape, 0, rng)
    values = _image("cont", shape, 0, rng)[:, 0].reshape(shape)
    near = _offsets_by_distance(min(100, (min(shape) - 2) // 4))
    nodes = []
    for _ in range(c["nodes"]):
        density = math.exp(rng.uniform(math.log(0.02), 0.0))
        sel = np.flatnonzero(rng.random(near.shape[0] - 1) < density)[:c["n"] - 1] + 1
        off = np.concatenate([np.zeros((1, 2), np.int32), near[sel]])
        at = rng.integers(0, shape[1]), rng.integers(0, shape[0])
        x = values[(at[1] + off[:, 1]) % shape[0], (at[0] + off[:, 0]) % shape[1]]
        u = np.stack([np.ones_like(x), x], 1)
        u[0] = 0.0
        d0 = float(-np.sum(x[1:].astype(np.float32) ** 2, dtype=np.float32))
        nodes.append((off, u.astype(np.float32), d0, float(rng.random())))
    return ti, nodes


def _grad_inputs(c, seed):
    """Features of encoder towers: (dx, dy, value) per slot, sparse for the
    queries, full for the keys; parameters as a fresh network holds them."""
    rng = np.random.default_rng([seed, 13])
    near = _offsets_by_distance(8)[1:g2s_lp.NB + 1].astype(np.float32) / 16.0

    def features(rows, cover):
        f = np.zeros((rows, g2s_lp.NB, 3), np.float32)
        base = rng.standard_normal((rows, 1))
        f[:, :, :2] = near
        f[:, :, 2] = base + 0.5 * rng.standard_normal((rows, g2s_lp.NB))
        f[rng.random((rows, g2s_lp.NB)) > cover] = 0.0
        return f.reshape(rows, g2s_lp.IN)

    params = []
    for _ in range(2):
        for din, dout in _LAYERS:
            params.append(rng.standard_normal(din * dout) * math.sqrt(2.0 / din))
            params.append(0.01 * rng.standard_normal(dout))
    return (np.concatenate(params).astype(np.float32), features(c["batch"], 0.6), features(c["keys"], 1.0))


_LAYERS = ((240, 256), (256, 256), (256, 256), (256, 128))
_INV_TAU = 10.0


def prepare(case, seed):
    c = dict(case)
    if c["family"] == "qs":
        return dict(c=c, q=_prepare_qs(c, seed))
    if c["family"] in ("wave", "node"):
        ti, nodes = _path_nodes(c, seed)
        dims = (c["x"], c["y"])
        image = g2s_amd.TrainingImage(g2s_amd.ti_subimages(ti, dims, [0]), dims)
        dev = g2s_amd.AcceleratorDevice(image, g2s_amd.coef_matrix([0])[0])
        s = dict(c=c, nodes=nodes, image=image, dev=dev)
        if c["family"] == "wave":
            s["wave"] = dev.wave(nodes, c["k"])
        return s
    if c["family"] == "calib":
        ti = _image("cont", (c["y"], c["x"]), 0, np.random.default_rng([seed, 14]))
        kd = (c["kernel"], c["kernel"])
        return dict(c=c, ti=ti, kernel=np.ones(kd[0] * kd[1], np.float32), kd=kd, seed=seed,
                    nb=g2s_amd.default_neighbour_configs((c["max_nb"],)))
    params, q, k = _grad_inputs(c, seed)
    net = g2s_lp.LearnedProposal()
    net.set_params(params)
    return dict(c=c, net=net, q=q, k=k)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    c = state["c"]
    if c["family"] == "qs":
        q = state["q"]
        sim, index, _ = g2s_amd.qs(q["ti"], q["ti_dims"], q["di"], q["sim_dims"], q["types"], q["n"], q["k"],
                                   q["seed"])
        return sim, index
    if c["family"] == "wave":
        state["wave"].run()
        return state["wave"].read()
    if c["family"] == "node":
        offsets, values, delta0, seed = state["nodes"][0]
        state["dev"].candidate_for_pattern(offsets, values, delta0)
        return state["dev"].search_k_biggest(int(math.ceil(c["k"])), seed)
    if c["family"] == "calib":
        r = g2s_amd.calibration([state["ti"]], (c["x"], c["y"]), [0], [state["kernel"]], [state["kd"]],
                                nb_configs=state["nb"], max_iter=c["iters"], seed=state["seed"])
        return r["mean"], r["dev"], r["samples"]
    loss, grad = state["net"].loss_grad(state["q"], state["k"], inv_tau=_INV_TAU)
    return float(loss), grad


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its result in 64 bits
# ---------------------------------------------------------------------------
def work(case):
    c = case
    if c["family"] == "qs":
        cells = int(np.prod(_dims(c)))
        sim = int(np.prod(_dims(c, "sx", "sy", "sz")))
        nvar = 2 if c["kind"] == "multi" else 1
        # every node scores every position of the image: one real inverse transform of the map
        return dict(bytes=4 * (cells * nvar + sim * (2 * nvar + 1)),
                    flops=sim * (1.0 - c["hard"]) * 2.5 * cells * math.log2(cells))
    if c["family"] in ("wave", "node"):
        cells, kk = c["x"] * c["y"], int(math.ceil(c["k"]))
        return dict(bytes=4 * 2 * cells + c["nodes"] * (c["n"] * 16 + 8 * kk + 4),
                    flops=c["nodes"] * 2.5 * cells * math.log2(cells))
    if c["family"] == "calib":
        cells, settings = c["x"] * c["y"], (c["max_nb"] - 1) * 7
        return dict(bytes=4 * (cells + c["kernel"] ** 2 + 3 * settings),
                    flops=settings * c["iters"] * 2.5 * cells * math.log2(cells))
    weights = sum(a * b for a, b in _LAYERS)
    rows = c["batch"] + c["keys"]
    return dict(bytes=4 * (rows * g2s_lp.IN + 4 * weights),
                flops=6.0 * rows * weights + 6.0 * c["batch"] * c["keys"] * g2s_lp.EMB)


def _exact_errors(c, seed):
    """Per node the K largest values of delta0 + sum_j (2 x_j y(p + d_j) - y(p + d_j)^2)."""
    ti, nodes = _path_nodes(c, seed)
    where = "cuda" if torch.cuda.is_available() else "cpu"
    y = torch.from_numpy(ti[:, 0].astype(np.float64).reshape(c["y"], c["x"])).to(where)
    y2 = torch.from_numpy((ti[:, 0] * ti[:, 0]).astype(np.float64).reshape(c["y"], c["x"])).to(where)
    kk = int(math.ceil(c["k"]))
    out = []
    for off, u, d0, _ in nodes:
        lo = [int(-min(0, off[:, d].min())) for d in range(2)]
        hi = [int(s - 1 - max(0, off[:, d].max())) for d, s in enumerate((c["x"], c["y"]))]
        acc = torch.full((hi[1] - lo[1] + 1, hi[0] - lo[0] + 1), float(np.float32(d0)), dtype=torch.float64,
                         device=where)
        for (a, b), (w, wx) in zip(off.tolist(), u.tolist()):
            if w == 0.0:
                continue
            part = slice(lo[1] + b, hi[1] + b + 1), slice(lo[0] + a, hi[0] + a + 1)
            acc += 2.0 * wx * y[part] - w * y2[part]
        out.append(torch.topk(acc.reshape(-1), kk).values.cpu().numpy())
    return np.stack(out)


def _exact_grad(c, seed):
    params, q, k = _grad_inputs(c, seed)
    p = torch.from_numpy(params.astype(np.float64)).requires_grad_(True)
    at = 0

    def tower(h):
        nonlocal at
        for i, (din, dout) in enumerate(_LAYERS):
            w = p[at:at + din * dout].reshape(din, dout)
            b = p[at + din * dout:at + din * dout + dout]
            at += din * dout + dout
            h = h @ w + b
            h = torch.relu(h) if i < 3 else h
        return h

    eq = tower(torch.from_numpy(q.astype(np.float64)))
    ek = tower(torch.from_numpy(k.astype(np.float64)))
    z = eq @ ek.T * _INV_TAU
    loss = torch.nn.functional.cross_entropy(z, torch.arange(z.shape[0]))
    loss.backward()
    return float(loss), p.grad.numpy()


def exact(case, seed):
    c = case
    if c["family"] == "wave":
        return _exact_errors(c, seed), None, None
    if c["family"] == "node":
        return _exact_errors(c, seed)[0], None
    if c["family"] == "grad":
        return _exact_grad(c, seed)
    # realisations and calibrations follow from chains of selections: in plain
    # 64-bit code they take minutes
    return None
