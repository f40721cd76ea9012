"""The data-flow path loop (tuning key loop.flow) against the wave loop, the
general path of the same realisation: identical bytes. The selection of both
is exact (FP64 values by the device rule, or whole counts under a tie quantum
that divides the weight), so no tolerance applies. The requests cover every
form that the data-flow loop takes: 1-3 dimensions, extents around the tile
and word edges (16, 32, 64), list lengths, weights, given and partially given
cells, images of n and k, several kernels, wrapping grids and images whose
best positions tie by the thousand."""
import numpy as np
import pytest

import g2s_amd

pytestmark = pytest.mark.gpu


def _field(dims, rng, kind):
    a = rng.standard_normal(tuple(reversed(dims)))
    for ax in range(a.ndim):
        a = a + np.roll(a, 1, ax) + 0.5 * np.roll(a, 2, ax)
    a = (a - a.mean()) / a.std()
    if kind == "cont":
        return np.exp(a).reshape(-1)
    if kind == "flat":
        return np.zeros(a.size)
    if kind == "steps":  # few distinct values: many exact ties
        return np.round(a).reshape(-1)
    return np.digitize(a, np.quantile(a, np.arange(1, int(kind)) / int(kind))).astype(float).reshape(-1)


def _both(*args, **kw):
    out = []
    try:
        for flow in (1, 0):
            g2s_amd.set_default_tuning("loop.flow", flow)
            s, i, st = g2s_amd.qs(*args, stage_timing=True, **kw)
            out.append((s.tobytes(), i.tobytes(), st))
    finally:
        g2s_amd.set_default_tuning("loop.flow", 1)
    assert out[0][0] == out[1][0] and out[0][1] == out[1][1]
    # the data-flow loop has no gather stage of its own
    assert out[0][2]["gather_ms"] == 0.0 < out[1][2]["gather_ms"] and out[0][2]["waves"] == out[1][2]["waves"]
    return out[0][2], out[1][2]


CASES = [
    # kinds per variable, image, grid, n, k, extra
    (("cont",), (300,), (120,), 9, 1.5, {}),
    (("cont",), (17, 5), (12, 9), 4, 1.0, {}),
    (("cont",), (64, 63), (31, 17), 12, 2.0, dict(hard=0.1)),
    (("cont",), (33, 129), (40, 13), 80, 3.0, dict(csim=True)),
    (("cont",), (37, 18, 9), (11, 7, 6), 25, 1.5, dict(hard=0.05)),
    (("cont",), (97, 65), (20, 20), 30, 16.0, dict(weights="distance")),
    (("cont",), (81, 70), (24, 20), 20, 1.5, dict(weights=0.5, nimg=True, kimg=True)),
    (("cont",), (60, 61), (20, 16), 14, 1.5, dict(kernels=True)),
    (("flat",), (48, 40), (10, 8), 6, 2.0, {}),
    (("steps",), (70, 52), (16, 16), 3, 1.5, {}),
    (("cont", "cont"), (55, 44), (18, 14), 16, 1.5, dict(partial=True)),
    (("cont", "3"), (66, 50), (20, 14), 18, 1.5, dict(hard=0.1, partial=True)),
    (("3", "cont"), (50, 41), (14, 12), 10, 1.2, {}),
    (("2",), (31, 20), (16, 13), 7, 1.0, {}),
    (("2",), (97, 33), (25, 21), 50, 1.2, dict(hard=0.1, csim=True)),
    (("4",), (65, 40), (20, 12), 150, 5.0, dict(weights=2.0)),
    (("3",), (40, 33, 12), (10, 9, 7), 40, 1.5, dict(kimg=True)),
    (("3",), (400,), (90,), 11, 1.5, {}),
    (("2", "3"), (60, 45), (15, 14), 20, 16.0, dict(partial=True, quantum=0.0)),
    # three and four variables, continuous ones among them
    (("cont", "3", "cont"), (52, 47), (14, 12), 15, 3.0, dict(partial=True, hard=0.05)),
    (("cont", "2", "cont", "3"), (40, 38), (12, 11), 9, 9.0, dict(weights="distance")),
    # several slices a node: counts, mixed
    (("2",), (250, 250), (40, 40), 50, 1.2, {}),
    (("cont", "4"), (200, 190), (24, 20), 40, 1.5, dict(hard=0.1)),
]


def _request(case):
    kinds, dims, sdims, n, k, x = CASES[case]
    print(f"data-flow loop: case {case} {CASES[case]}", flush=True)
    rng = np.random.default_rng(100 + case)
    types = [0 if q in ("cont", "flat", "steps") else 1 for q in kinds]
    ti = np.stack([_field(dims, rng, q) for q in kinds], 1).astype(np.float32)
    cells = int(np.prod(sdims))
    di = np.full((cells, len(kinds)), np.nan, np.float32)
    u = rng.random(cells)
    src = ti[rng.integers(0, ti.shape[0], cells)]
    if "hard" in x:
        di[u < x["hard"]] = src[u < x["hard"]]
    if "partial" in x:
        one = u > 0.8
        di[one, case % len(kinds)] = src[one, case % len(kinds)]
    kd = [d // 2 + 1 for d in dims]
    kw = dict(circular_sim=x.get("csim", False), tie_quantum=x.get("quantum", -1.0))
    if "weights" in x:
        if x["weights"] == "distance":
            ker = g2s_amd.kernel_generate(kd, [2] * len(kinds), [1.0] * len(kinds), [0.05] * len(kinds))
        else:
            ker = np.full(int(np.prod(kd)) * len(kinds), x["weights"], np.float32)
        kw.update(kernel=ker, kernel_dims=kd)
    if "nimg" in x:
        kw["n_image"] = rng.integers(0, n + 1, cells).astype(np.float32)
    if "kimg" in x:
        kw["k_image"] = rng.choice([1.0, k, 2.5], cells).astype(np.float32)
    if "kernels" in x:
        sizes = [kd, [9, 11]]
        kw.update(kernels=[np.ones(int(np.prod(s)), np.float32) for s in sizes], kernels_dims=sizes,
                  kernel_index_image=rng.integers(0, 2, cells).astype(np.float32))
    return (ti, dims, di, sdims, types, n, k, 5 + case), kw


@pytest.mark.parametrize("case", range(len(CASES)))
def test_flow_equals_waves(case):
    args, kw = _request(case)
    _both(*args, **kw)


@pytest.mark.parametrize("case", range(len(CASES)))
def test_flow_then_waves(case):
    """The path handed over in the middle, at a place that cuts a level."""
    args, kw = _request(case)
    try:
        g2s_amd.set_default_tuning("flow.nodes", int(np.prod(CASES[case][2])) // 3)
        a = g2s_amd.qs(*args, stage_timing=True, **kw)
        g2s_amd.set_default_tuning("loop.flow", 0)
        b = g2s_amd.qs(*args, **kw)
    finally:
        g2s_amd.set_default_tuning("flow.nodes", 0)
        g2s_amd.set_default_tuning("loop.flow", 1)
    assert a[0].tobytes() == b[0].tobytes() and a[1].tobytes() == b[1].tobytes()
    assert a[2]["gather_ms"] > 0.0 and a[2]["waves"] == b[2]["waves"]


@pytest.mark.parametrize("kind", ["cont", "3"])
def test_flow_without_valid_position(kind):
    """Kernels larger than the image: many nodes have no position whose
    neighbours all lie inside it; their cells stay empty and give their
    neighbours nothing."""
    rng = np.random.default_rng(17)
    dims, sdims, kd = (9, 7), (25, 20), [21, 21]
    ti = _field(dims, rng, kind).astype(np.float32)
    di = np.full(int(np.prod(sdims)), np.nan, np.float32)
    kw = dict(kernel=np.ones(kd[0] * kd[1], np.float32), kernel_dims=kd)
    args = (ti, dims, di, sdims, [0 if kind == "cont" else 1], 6, 2.0, 3)
    _both(*args, **kw)
    empty = int(np.isnan(g2s_amd.qs(*args, **kw)[0]).sum())
    print(f"data-flow loop: {empty} of {di.size} cells without a valid position", flush=True)
    assert 0 < empty < di.size


def test_flow_without_memory_for_waves():
    """A hand-over to waves that do not fit (levels of 100,000 nodes of a 1000
    x 1000 image, 8 MB each): the data-flow loop simulates the whole path."""
    rng = np.random.default_rng(19)
    dims, sdims = (1000, 1000), (1000, 1000)
    args = (_field(dims, rng, "cont").astype(np.float32), dims, np.full(sdims[0] * sdims[1], np.nan, np.float32),
            sdims, [0], 2, 1.0, 3)
    out = []
    try:
        for nodes in (0, 1000):
            g2s_amd.set_default_tuning("flow.nodes", nodes)
            out.append(g2s_amd.qs(*args, wave_size=1 << 20, stage_timing=True))
    finally:
        g2s_amd.set_default_tuning("flow.nodes", 0)
    assert out[0][0].tobytes() == out[1][0].tobytes() and out[0][1].tobytes() == out[1][1].tobytes()
    assert out[0][2]["gather_ms"] == out[1][2]["gather_ms"] == 0.0


def test_flow_slices_and_segments():
    """An image large enough for several slices a node and a path of several
    launches (64 nodes in flight, 64 x 64 a launch)."""
    rng = np.random.default_rng(3)
    dims, sdims = (410, 390), (80, 70)
    ti = _field(dims, rng, "cont").astype(np.float32)
    di = np.full(int(np.prod(sdims)), np.nan, np.float32)
    flow, waves = _both(ti, dims, di, sdims, [0], 24, 1.5, 4, wave_size=64)
    assert flow["exact_nodes"] == waves["exact_nodes"]


@pytest.mark.parametrize("n,default,finer", [(50, -10, 0), (50, -10, 1), (300, -7, 9)])
def test_flow_tie_quantum(n, default, finer):
    """A tie quantum finer than the default (2^default for n neighbours of
    weight 1) may be less than twice the FP32 map's error (2^-16 is less than
    the spacing of FP32 numbers at 300): the wave loop's selection is what the
    request gets then."""
    rng = np.random.default_rng(31)
    dims, sdims = (250, 250), (40, 36)
    ti = _field(dims, rng, "2").astype(np.float32)
    di = np.full(int(np.prod(sdims)), np.nan, np.float32)
    out = []
    try:
        for flow in (1, 0):
            g2s_amd.set_default_tuning("loop.flow", flow)
            out.append(g2s_amd.qs(ti, dims, di, sdims, [1], n, 1.2, 3, tie_quantum=2.0 ** (default - finer),
                                  stage_timing=True))
    finally:
        g2s_amd.set_default_tuning("loop.flow", 1)
    assert out[0][0].tobytes() == out[1][0].tobytes() and out[0][1].tobytes() == out[1][1].tobytes()
    assert (out[0][2]["gather_ms"] > 0.0) == (finer > 0)


@pytest.mark.parametrize("kinds", [("cont",), ("3",), ("cont", "3")])
def test_flow_gives_up(kinds):
    """A wait that hits its bound (here the first poll that finds a value
    missing) ends the loop; the wave loop simulates the path from its start."""
    rng = np.random.default_rng(21)
    dims, sdims = (150, 140), (30, 26)
    ti = np.stack([_field(dims, rng, q) for q in kinds], 1).astype(np.float32)
    di = np.full((int(np.prod(sdims)), len(kinds)), np.nan, np.float32)
    types = [0 if q == "cont" else 1 for q in kinds]
    out = []
    try:
        for key, value in (("flow.polls", 1), ("loop.flow", 0)):
            g2s_amd.set_default_tuning(key, value)
            out.append(g2s_amd.qs(ti, dims, di, sdims, types, 40, 1.5, 2, stage_timing=True))
            g2s_amd.set_default_tuning("flow.polls", 0)
    finally:
        g2s_amd.set_default_tuning("loop.flow", 1)
        g2s_amd.set_default_tuning("flow.polls", 0)
    for a, b in zip(out[0][:2], out[1][:2]):
        assert a.tobytes() == b.tobytes()
    assert out[0][2]["gather_ms"] > 0.0


def test_flow_gives_up_at_once():
    """What is left of the path after a given-up wait is not simulated: on an
    image where the data-flow loop takes longer than the waves (white noise,
    250 neighbours, 10 best), the run costs little more than the waves alone.
    Half of their time is room for the first nodes and the timer; the rest of
    the path would take more than all of it."""
    rng = np.random.default_rng(22)
    dims, sdims = (1000, 1000), (100, 100)
    ti = rng.standard_normal(dims[0] * dims[1]).astype(np.float32)
    di = np.full(sdims[0] * sdims[1], np.nan, np.float32)
    ms = {}
    try:
        for name, key, value in (("warm", "loop.flow", 0), ("waves", "loop.flow", 0), ("given up", "flow.polls", 1)):
            g2s_amd.set_default_tuning("loop.flow", 1)
            g2s_amd.set_default_tuning(key, value)
            ms[name] = g2s_amd.qs(ti, dims, di, sdims, [0], 250, 10.0, 6)[2]["path_loop_ms"]
            print(f"data-flow loop: {name} {ms[name]:.0f} ms", flush=True)
    finally:
        g2s_amd.set_default_tuning("loop.flow", 1)
        g2s_amd.set_default_tuning("flow.polls", 0)
    assert ms["given up"] < 1.5 * ms["waves"]


@pytest.mark.parametrize("kinds,n,k,sdims,over", [
    (("noise",), 80, 1.5, (530, 500), True),
    (("noise",), 250, 1.5, (120, 120), True),
    (("noise", "noise"), 60, 1.5, (100, 100), True),
    (("noise",), 80, 10.0, (120, 120), True),
    (("cont",), 80, 1.5, (150, 150), False),
    (("zeros",), 80, 10.0, (100, 100), False),
])
def test_flow_hands_over_to_waves(kinds, n, k, sdims, over):
    """1000 x 1000 images: white noise, where the wave loop takes over the rest
    of the path, a smooth image and one of mostly zeros (whose ties overflow
    the wave loop's lists), where it does not."""
    rng = np.random.default_rng(8)
    dims = (1000, 1000)
    ti = [rng.standard_normal(dims[0] * dims[1]) if q == "noise" else
          np.maximum(_field(dims, rng, "cont") - 5.0, 0.0) if q == "zeros" else _field(dims, rng, q) for q in kinds]
    ti = np.stack(ti, 1).astype(np.float32)
    di = np.full((sdims[0] * sdims[1], len(kinds)), np.nan, np.float32)
    out = []
    try:
        for flow in (1, 0):
            g2s_amd.set_default_tuning("loop.flow", flow)
            out.append(g2s_amd.qs(ti, dims, di, sdims, [0] * len(kinds), n, k, 6, stage_timing=True))
    finally:
        g2s_amd.set_default_tuning("loop.flow", 1)
    assert out[0][0].tobytes() == out[1][0].tobytes() and out[0][1].tobytes() == out[1][1].tobytes()
    assert out[0][2]["exact_nodes"] == out[1][2]["exact_nodes"]
    # only the wave loop has a gather stage; less of it where it came in later
    assert (0.0 < out[0][2]["gather_ms"] < out[1][2]["gather_ms"]) if over else out[0][2]["gather_ms"] == 0.0
