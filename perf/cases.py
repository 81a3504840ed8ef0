"""The filter's work as a program has it done, for timing: single filters from
the smallest online tracker to two million particles, batches of independent
filters, and served tracks, each through esthera_amd's own entry points.

A pass of a single filter is a stretch of its trace: one step per measurement,
an estimate every `every` steps (1: a tracker that acts on each one), then the
particles.  A batch's pass is a stretch of steps and every filter's estimate.
A server's pass is `rounds` updates of every open track, each round waited for.
Traces are closed loops (of ROWS measurements, in a batch of 8), so that a
filter can follow one for as long as it is run.
"""
import ctypes
import gc
import math
import os

import numpy as np

import esthera_amd as ea
from esthera_amd import workloads

ROWS = 64
MODELS = {"robotarm5": ea.MODEL_ROBOTARM5, "unicycle": ea.MODEL_UNICYCLE, "dh6": ea.MODEL_DH6,
          "unicycle10": ea.MODEL_UNICYCLE10, "robotarm5_camera": ea.MODEL_ROBOTARM5_CAMERA,
          "randomwalk3": ea.MODEL_RANDOMWALK3}
TOPOLOGIES = {"none": ea.TOPO_NONE, "ring": ea.TOPO_RING, "torus": ea.TOPO_TORUS, "all2all": ea.TOPO_ALL2ALL}
RESAMPLERS = {"multinomial": ea.RESAMPLE_MULTINOMIAL, "systematic": ea.RESAMPLE_SYSTEMATIC, "alias": ea.RESAMPLE_ALIAS}
LAYOUTS = {"soa": ea.LAYOUT_SOA, "aos": ea.LAYOUT_AOS, "packed": ea.LAYOUT_PACKED}
# arithmetic of one particle's propagation and likelihood, Box-Muller included
# (an FMA counts two); the unicycle's is per landmark beyond this
FLOPS = {"robotarm5": 650, "unicycle": 200, "dh6": 640, "unicycle10": 300, "robotarm5_camera": 700, "randomwalk3": 130}
FLOPS_LANDMARK = 80


def _filter(model, m, G, t, topology, resampler, weights, steps, every, landmarks=0, threshold=1.0, adaptive=0, carry=0,
            layout="soa"):
    return {"kind": "filter", "model": model, "m": m, "G": G, "t": t, "topology": topology, "resampler": resampler,
            "weights": weights, "steps": steps, "every": every, "landmarks": landmarks, "threshold": threshold,
            "adaptive": adaptive, "carry": carry, "layout": layout}


def listed():
    return [
        # the reference driver's own setting (its robot arm, few and small sub-filters, linear weights, multinomial
        # selection), the estimate read after every step: launches and latency are everything
        dict(_filter("robotarm5", 64, 16, 1, "ring", "multinomial", "linear", 32, 1), name="arm_64x16_online"),
        # the accuracy workload: 4096 particles, 4 landmarks, read after every step
        dict(_filter("unicycle", 256, 16, 1, "torus", "systematic", "log", 32, 1, 4), name="unicycle_256x16_online"),
        # a tracker of a quarter of a million particles over the reference's ten range sensors; the gate leaves half of
        # the sub-filters, whose number is no power of two, unresampled in each step
        dict(_filter("unicycle10", 256, 1000, 2, "ring", "alias", "log", 32, 1, threshold=0.5),
             name="unicycle10_256x1000_alias"),
        # many small sub-filters with a cheap likelihood and an odd count
        dict(_filter("randomwalk3", 128, 3001, 1, "ring", "multinomial", "log", 64, 8), name="walk_128x3001"),
        # the headline workload, streamed over its trace as in offline estimation
        dict(_filter("unicycle", 512, 4096, 4, "torus", "systematic", "log", 200, 100, 32), name="unicycle_512x4096"),
        # the same filter acting on every estimate
        dict(_filter("unicycle", 512, 4096, 4, "torus", "systematic", "log", 100, 1, 32), name="unicycle_512x4096_online"),
        # its other resampler
        dict(_filter("unicycle", 512, 4096, 4, "torus", "alias", "log", 200, 100, 32), name="unicycle_512x4096_alias"),
        # the same particles with few landmarks, where memory counts
        dict(_filter("unicycle", 512, 4096, 4, "torus", "systematic", "log", 200, 100, 4), name="unicycle_512x4096_4lm"),
        # the six-joint arm: twelve state variables
        dict(_filter("dh6", 512, 2048, 1, "torus", "systematic", "log", 200, 100), name="dh6_512x2048"),
        # the largest sub-filters, nine state variables, the global best exchanged
        dict(_filter("robotarm5", 1024, 500, 4, "all2all", "multinomial", "log", 100, 20), name="arm_1024x500"),
        # ten thousand independent filters of 256 to 65536 particles in one batch (118.8 M particles)
        {"name": "batch_10000", "kind": "batch", "filters": 10000, "landmarks": 8, "steps": 100},
        # tracks of 1024 to 262144 particles, seven of ten unicycles and three robot arms, updated as one wave after another
        {"name": "served_256", "kind": "server", "tracks": 256, "landmarks": 8, "rounds": 8},
    ]


def draw(rng):
    """One more case of the same ranges: every model, sub-filters of 16 to 1024 particles in any number up to two
    million particles in all, every exchange, resampler, weighting and layout; batches and servers of any size up to
    the listed ones."""
    what = rng.random()
    if what < 0.12:
        n = int(round(math.exp(rng.uniform(math.log(16), math.log(4000)))))
        return {"kind": "batch", "filters": n, "landmarks": rng.choice([4, 8, 8, 16]), "steps": rng.randint(20, 40)}
    if what < 0.22:
        return {"kind": "server", "tracks": int(round(math.exp(rng.uniform(math.log(2), math.log(256))))),
                "landmarks": rng.choice([4, 8, 8, 16]), "rounds": rng.randint(4, 8)}
    model = rng.choice(["unicycle", "unicycle", "unicycle", "unicycle10", "randomwalk3", "robotarm5", "robotarm5",
                        "robotarm5_camera", "dh6"])
    S = ea.STATE_DIM[MODELS[model]]
    m = rng.choice([16, 32, 64, 64, 128, 128, 256, 256, 512, 512, 512, 1024])
    most = min(8192, (2097152 if S == 3 else 1048576) // m)
    G = max(2, int(round(math.exp(rng.uniform(math.log(8), math.log(most))))))
    topology = rng.choice(["none", "ring", "ring", "torus", "torus", "torus", "all2all"])
    if topology == "torus":   # a torus of whole rows
        G = max(4, G - G % (1 << int(math.log2(math.sqrt(G)))))
    t = 0 if topology == "none" else rng.choice([1, 1, 2, 4])
    weights = rng.choice(["log", "log", "log", "linear"])
    resampler = rng.choice(["systematic", "systematic", "multinomial", "alias"])
    steps = max(16, min(64, int(2.0e7 / (m * G))))
    return _filter(model, m, G, t, topology, resampler, weights, steps, rng.choice([1, 1, 8, steps]),
                   rng.choice([2, 4, 8, 13, 20, 32]) if model == "unicycle" else 0, rng.choice([1.0, 1.0, 1.0, 0.5, 0.8]),
                   0, 1 if rng.random() < 0.1 else 0, rng.choice(["soa"] * 8 + ["aos", "packed"]))


# ------------------------------------------------------------------ traces
def _loop(v, omega, rows):
    """Steps of 0.1 s along a regular polygon: positions and headings after each, from (0, 0) and heading 0."""
    k = np.arange(rows)
    step = v * 0.1 * np.stack([np.cos(omega * 0.1 * k), np.sin(omega * 0.1 * k)], 1)
    return np.cumsum(step, 0), omega * 0.1 * (k + 1)


def _arm_camera_point(q, x, y):
    """The base in the arm's camera frame (rows of angles q)."""
    X = x * np.cos(q[:, 0]) + y * np.sin(q[:, 0])
    Y = -x * np.sin(q[:, 0]) + y * np.cos(q[:, 0])
    Z = np.zeros_like(X)
    for i in range(1, 5):
        Y, Z = Y * np.cos(q[:, i]) - Z * np.sin(q[:, i]), Y * np.sin(q[:, i]) + Z * np.cos(q[:, i]) - 3.0
    return X, Y, Z


def _trace(model, landmarks, seed, rows=ROWS):
    """A closed trace: parameters, controls and measurements of each row, the time step, the state before the first
    step and the spread of the particles around it."""
    rng = np.random.default_rng([seed, 7])
    turn = 2 * math.pi * np.arange(rows) / rows
    ctrl, meas = [], []
    if model == "unicycle":
        box = 0.0 if landmarks == 4 else 20.0 if landmarks < 16 else 50.0
        params = ea.unicycle_scenario(seed, landmarks, box, 0)[0]
        omega = 2 * math.pi / (rows * 0.1)
        at, th = _loop(1.0, omega, rows)
        for k in range(rows):
            c, z = ea.UnicycleControl(1.0, omega), ea.UnicycleMeasurement()
            d = np.stack([params.lx[:landmarks], params.ly[:landmarks]], 1) - at[k]
            z.range[:landmarks] = np.hypot(d[:, 0], d[:, 1]) + 0.1 * rng.standard_normal(landmarks)
            b = np.arctan2(d[:, 1], d[:, 0]) - th[k] + 0.02 * rng.standard_normal(landmarks)
            z.bearing[:landmarks] = np.arctan2(np.sin(b), np.cos(b))
            ctrl.append(c), meas.append(z)
        return params, ctrl, meas, 0.1, np.zeros(3), np.array([0.2, 0.2, 0.05])
    if model == "unicycle10":
        params = ea.unicycle10_params_default()
        omega = 2 * math.pi / (rows * 0.1)
        at, th = _loop(2.0, omega, rows)
        sensors = np.stack([params.sx, params.sy, params.sz], 1)
        for k in range(rows):
            p = np.array([16.0 + at[k, 0], 24.0 + at[k, 1], 0.0])
            z = ea.Unicycle10Measurement()
            z.range[:] = np.linalg.norm(sensors - p, axis=1) + 0.3 * rng.standard_normal(10)
            ctrl.append(ea.UnicycleControl(2.0, omega)), meas.append(z)
        return params, ctrl, meas, 0.1, np.array([16.0, 24.0, 0.0]), np.array([0.5, 0.5, 0.1])
    if model == "randomwalk3":
        params = ea.RandomWalk3Params(0.05, 0.2)
        v = np.stack([np.cos(turn), np.sin(turn), np.cos(2 * turn)], 1)
        at = np.cumsum(v * 0.1, 0)
        for k in range(rows):
            c, z = ea.RandomWalk3Control(), ea.RandomWalk3Measurement()
            c.v[:] = v[k]
            z.p[:] = at[k] + 0.2 * rng.standard_normal(3)
            ctrl.append(c), meas.append(z)
        return params, ctrl, meas, 0.1, np.zeros(3), np.full(3, 0.3)
    if model == "dh6":
        params = ea.dh6_scenario(seed, 0)[0]
        dt, amp, phase = 0.01, 0.01 * rng.uniform(0.2, 1.0, 6), rng.uniform(0, 2 * math.pi, 6)
        rest, w = rng.uniform(-0.5, 0.5, 6), 2 * math.pi / (rows * dt)
        q = rest + amp * np.sin(turn[:, None] + 2 * math.pi / rows + phase)
        p = np.zeros((rows, 3))
        for i in range(5, -1, -1):
            ca, sa, cq, sq = math.cos(params.alpha[i]), math.sin(params.alpha[i]), np.cos(q[:, i]), np.sin(q[:, i])
            u, side = p[:, 0] + params.a[i], ca * p[:, 1] - sa * p[:, 2]
            p = np.stack([cq * u - sq * side, sq * u + cq * side, sa * p[:, 1] + ca * p[:, 2] + params.d[i]], 1)
        for k in range(rows):
            z = ea.DH6Measurement()
            z.p[:] = p[k] + 0.01 * rng.standard_normal(3)
            z.q[:] = q[k] + 0.005 * rng.standard_normal(6)
            ctrl.append(ea.DH6Control(0.0)), meas.append(z)
        start = np.concatenate([rest + amp * np.sin(phase), amp * w * np.cos(phase)])
        return params, ctrl, meas, dt, start, np.repeat([0.01, 0.05], 6)
    # the robot arms: joints swing about their rest, the base stands still
    phase, base = rng.uniform(0, 2 * math.pi, 5), np.array([0.5, -0.4])
    rate = 0.2 * np.cos(turn[:, None] + phase)
    q = 0.75 * math.pi + np.cumsum(rate * 0.1, 0)
    X, Y, Z = _arm_camera_point(q, *base)
    params = None
    if model == "robotarm5_camera":
        params = ea.camera_params_default()
        fc, cc, kc = params.fc, params.cc, params.kc
        xn, yn = X / Z, Y / Z
        r2 = xn * xn + yn * yn
        k1 = 1 + kc[0] * r2 + kc[1] * r2 * r2
        X = fc[0] * (k1 * xn + 2 * kc[2] * xn * yn + kc[3] * (r2 + 2 * xn * xn)) + cc[0]
        Y = fc[1] * (k1 * yn + kc[2] * (r2 + 2 * yn * yn) + 2 * kc[3] * xn * yn) + cc[1]
    for k in range(rows):
        c, z = ea.RobotArm5Control(), ea.RobotArm5Measurement()
        c.angles[:] = rate[k]
        z.angles[:] = q[k] + 0.05 * rng.standard_normal(5)
        z.x, z.y = X[k] + 0.1 * rng.standard_normal(), Y[k] + 0.1 * rng.standard_normal()
        ctrl.append(c), meas.append(z)
    start = np.concatenate([np.full(5, 0.75 * math.pi), base, np.zeros(2)])
    return params, ctrl, meas, 0.1, start, np.array([0.1] * 5 + [0.2] * 4)


def _start(case, seed, start, spread):
    """The first particles: S planes of m G floats."""
    n = case["m"] * case["G"]
    z = np.random.default_rng([seed, 11]).standard_normal((len(start), n), dtype=np.float32)
    return z * spread[:, None].astype(np.float32) + start[:, None].astype(np.float32)


# ------------------------------------------------------------------- cases
_ENGINE = None


def _engine():
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = ea.Engine(0)
        # batches: two sub-filters of 64 to a wave, as the autotuner sets it
        _ENGINE.set_batch_resample_lanes(64, 32)
    gc.collect()   # filters of earlier states return their memory
    return _ENGINE


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)
        self.k = 0


def prepare(case, seed):
    return {"filter": _prepare_filter, "batch": _prepare_batch, "server": _prepare_server}[case["kind"]](case, seed)


def run(state):
    return state.run(state)


def _prepare_filter(case, seed):
    params, ctrl, meas, dt, start, spread = _trace(case["model"], case["landmarks"], seed)
    desc = ea.filter_desc(MODELS[case["model"]], m=case["m"], G=case["G"], t=case["t"],
                          topology=TOPOLOGIES[case["topology"]], resampler=RESAMPLERS[case["resampler"]],
                          threshold=case["threshold"], adaptive=case["adaptive"],
                          weights=ea.WEIGHTS_LOG if case["weights"] == "log" else ea.WEIGHTS_LINEAR,
                          seed=seed % 1000003, carry=case["carry"], layout=LAYOUTS[case["layout"]])
    f = ea.Filter(_engine(), desc, params)
    f.init(_start(case, seed, start, spread))
    return _State(run=_run_filter, f=f, ctrl=ctrl, meas=meas, dt=dt, steps=case["steps"], every=case["every"])


def _estimates(es):
    """Estimates as arrays: posterior means, best particles, [log weight maximum, weight sum, best weight], sub-filter
    of the best."""
    S = es[0].state_dim
    return {"mean": np.array([e.mean[:S] for e in es]), "best": np.array([e.best[:S] for e in es], np.float32),
            "weight": np.array([(e.log_weight_max, e.weight_sum, e.best_weight) for e in es]),
            "block": np.array([e.best_block for e in es], np.int64)}


def _run_filter(s):
    f, es = s.f, []
    for i in range(s.steps):
        f.step(s.ctrl[s.k], s.meas[s.k], s.dt)
        s.k = (s.k + 1) % ROWS
        if i % s.every == 0:
            es.append(f.estimate())
    es.append(f.estimate())
    particles, weights = f.particles()
    return {"first": _estimates(es[:1]), "later": _estimates(es[1:]), "particles": particles, "weights": weights}


def _prepare_batch(case, seed):
    n, L = case["filters"], case["landmarks"]
    traces = [_trace("unicycle", L, seed * 64 + j, 8) for j in range(min(64, n))]
    scen = [(t[0], t[1], t[2]) for t in traces]
    # sub-filters as large as the count's factors of two allow, up to the 128 that measures best
    counts, descs, params, _ = workloads.batched_filters(None, n, 99, scen, lambda c: min(128, c & -c))
    for i, d in enumerate(descs):
        d.seed = (seed * 1009 + i * 7919) % (1 << 31)
    b = ea.Batch(_engine(), descs, params)
    b.init_uniform(np.random.default_rng([seed, 13]).normal(0.0, 0.05, (n, 3)).astype(np.float32))
    ctrl = [(ea.UnicycleControl * n)(*[scen[i % len(scen)][1][k] for i in range(n)]) for k in range(8)]
    meas = [(ea.UnicycleMeasurement * n)(*[scen[i % len(scen)][2][k] for i in range(n)]) for k in range(8)]
    return _State(run=_run_batch, b=b, n=n, ctrl=ctrl, meas=meas, dts=np.full(n, 0.1, np.float32), steps=case["steps"])


def _run_batch(s):
    for _ in range(s.steps):
        s.b.step(s.ctrl[s.k], s.meas[s.k], s.dts)
        s.k = (s.k + 1) % len(s.ctrl)
    return _estimates([s.b.estimate(i) for i in range(s.n)])


def _prepare_server(case, seed):
    n = case["tracks"]
    rng = np.random.default_rng([seed, 17])
    sizes = np.exp(np.random.default_rng(5).uniform(math.log(1024), math.log(262144), n))
    s = ea.Server(_engine(), n, 32 << 30)
    kinds = [_trace("unicycle", case["landmarks"], seed * 64 + j) for j in range(7)]
    kinds += [_trace("robotarm5", 0, seed * 64 + j) for j in range(3)]
    tracks = []
    for i in range(n):
        params, ctrl, meas, dt, start, spread = kinds[i % 10]
        arm = params is None
        m = 256 if sizes[i] < 16384 else 512
        d = ea.filter_desc(ea.MODEL_ROBOTARM5 if arm else ea.MODEL_UNICYCLE, m=m, G=max(2, int(sizes[i]) // m), t=1,
                           topology=ea.TOPO_RING, resampler=ea.RESAMPLE_SYSTEMATIC, weights=ea.WEIGHTS_LOG,
                           rng=ea.RNG_MTGP_PER_FILTER, seed=int(rng.integers(1 << 30)))
        tid, _ = s.open(d, params, start + spread * rng.normal(0.0, 0.1, len(start)))
        tracks.append((tid, ctrl, meas, dt))
    s.drain()
    s.poll(2 * n)
    return _State(run=_run_server, s=s, tracks=tracks, rounds=case["rounds"])


def _run_server(s):
    got = []
    for _ in range(s.rounds):
        for tid, ctrl, meas, dt in s.tracks:
            s.s.update(tid, ctrl[s.k], meas[s.k], dt)
        s.s.drain()
        got.append(sorted(s.s.poll(len(s.tracks) + 8), key=lambda r: r.request_id))
        s.k = (s.k + 1) % ROWS
    es = [r.estimate for g in got for r in g]
    S = max(e.state_dim for e in es)
    return {"mean": np.array([e.mean[:S] for e in es]), "best": np.array([e.best[:S] for e in es], np.float32),
            "weight": np.array([(e.log_weight_max, e.weight_sum, e.best_weight) for e in es]),
            "block": np.array([e.best_block for e in es], np.int64),
            "status": np.array([r.status for g in got for r in g], np.int64)}


def work(case):
    """Per step each particle's state is read and written once, its weight written once, its arithmetic done once, and
    its sub-filter ordered (m log2 m compares); the random numbers need no memory."""
    def of(model, landmarks, n, m, steps):
        S = ea.STATE_DIM[MODELS[model]]
        flops = FLOPS[model] + FLOPS_LANDMARK * landmarks + int(math.log2(m))
        return np.array([(8.0 * S + 4.0) * n * steps, float(flops) * n * steps])

    if case["kind"] == "filter":
        w = of(case["model"], case["landmarks"], case["m"] * case["G"], case["m"], case["steps"])
    elif case["kind"] == "batch":
        w = of("unicycle", case["landmarks"], int(workloads.batched_counts(case["filters"], 99).sum()), 128, case["steps"])
    else:
        w = np.zeros(2)
        sizes = np.exp(np.random.default_rng(5).uniform(math.log(1024), math.log(262144), case["tracks"]))
        for i, n in enumerate(sizes):
            arm = i % 10 >= 7
            w += of("robotarm5" if arm else "unicycle", 0 if arm else case["landmarks"], int(n), 256, case["rounds"])
    return {"bytes": float(w[0]), "flops": float(w[1])}


# ------------------------------------------------- the first step in 64 bits
def _mtgp_words(seed, K, size):
    """The words of K MTGP32 streams (parameter sets 0 .. K - 1, stream j seeded seed + j + 1), `size` each, as floats
    in [1, 2): the published recursion over the authors' table."""
    table = os.path.join(os.path.dirname(ea.__file__), "data", "mtgp32dc_11213.txt")
    with open(table) as fh:
        rows = [r.split() for r in fh if r.strip() and not r.startswith("#")]
    out = np.empty((K, size), np.float32)
    mask = np.uint32(int(rows[0][3], 16))
    for j in range(K):
        pos, sh1, sh2 = int(rows[j][0]), int(rows[j][1]), int(rows[j][2])
        t = np.array([int(x, 16) for x in rows[j][4:]], np.uint32)
        hidden = int(t[4]) ^ (int(t[8]) << 16 & 0xFFFFFFFF)
        fill = hidden + (hidden >> 16) & 0xFFFFFFFF
        fill = fill + (fill >> 8) & 0xFF
        x = np.full(351 + size, fill * 0x01010101, np.uint32)
        x[0], x[1] = (seed + j + 1) & 0xFFFFFFFF, hidden
        for i in range(1, 351):
            p = int(x[i - 1])
            x[i] = int(x[i]) ^ (1812433253 * (p ^ p >> 30) + i & 0xFFFFFFFF)
        most = 351 - pos
        for n in range(351, 351 + size, most):
            e = min(n + most, 351 + size)
            X = (x[n - 351:e - 351] & mask) ^ x[n - 350:e - 350]
            X ^= X << np.uint32(sh1)
            Y = X ^ (x[n - 351 + pos:e - 351 + pos] >> np.uint32(sh2))
            x[n:e] = Y ^ t[Y & 15]
        T = x[pos - 1:pos - 1 + size]
        T = T ^ T >> np.uint32(16)
        T = T ^ T >> np.uint32(8)
        out[j] = ((x[351:] >> np.uint32(9)) ^ t[32 + (T & 15)]).view(np.float32)
    return out.reshape(-1)


def _normals(words, n, V):
    """Box-Muller over consecutive pairs: V rows of n normals."""
    u = 2.0 - words[:V * n].astype(np.float64).reshape(V, n // 2, 2)
    r, phi = np.sqrt(-2.0 * np.log(u[..., 0])), 2.0 * math.pi * u[..., 1]
    return np.stack([r * np.cos(phi), r * np.sin(phi)], -1).reshape(V, n)


def _weigh(model, s, z, p, c, m, dt):
    """The propagated states and log weights of a model's step in 64 bits."""
    if model == "unicycle":
        x = s[0] + c.v * dt * np.cos(s[2]) + p.sigma_x * z[0]
        y = s[1] + c.v * dt * np.sin(s[2]) + p.sigma_y * z[1]
        th = s[2] + c.omega * dt + p.sigma_theta * z[2]
        lw = np.zeros_like(x)
        for j in range(p.num_landmarks):
            dx, dy = p.lx[j] - x, p.ly[j] - y
            b = m.bearing[j] - (np.arctan2(dy, dx) - th)
            b -= 2 * math.pi * np.rint(b / (2 * math.pi))
            lw -= 0.5 * (((m.range[j] - np.hypot(dx, dy)) / p.sigma_range) ** 2 + (b / p.sigma_bearing) ** 2)
        return np.stack([x, y, th]), lw
    if model == "unicycle10":
        v, w = c.v + p.noise_v * z[0], c.omega + p.noise_omega * z[1]
        h = 0.5 * w * dt
        chord = v * dt * np.sinc(h / math.pi)
        x, y = s[0] + chord * np.cos(s[2] + h), s[1] + chord * np.sin(s[2] + h)
        lw = np.full_like(x, math.log(1e5) - 5 * math.log(2 * math.pi))
        for j in range(10):
            lw -= (np.sqrt((x - p.sx[j]) ** 2 + (y - p.sy[j]) ** 2 + p.sz[j] ** 2) - m.range[j]) ** 2
        return np.stack([x, y, s[2] + w * dt + p.noise_gamma * z[2] * dt]), lw
    if model == "randomwalk3":
        x = s + dt * np.array(c.v[:])[:, None] + p.sigma_q * z
        return x, -0.5 * (((np.array(m.p[:])[:, None] - x) / p.sigma_r) ** 2).sum(0)
    if model == "dh6":
        a = p.sigma_acc * z
        q, qd = s[:6] + s[6:] * dt + 0.5 * dt * dt * a, s[6:] + a * dt
        e = np.zeros((3, q.shape[1]))
        for i in range(5, -1, -1):
            ca, sa, cq, sq = math.cos(p.alpha[i]), math.sin(p.alpha[i]), np.cos(q[i]), np.sin(q[i])
            u, side = e[0] + p.a[i], ca * e[1] - sa * e[2]
            e = np.stack([cq * u - sq * side, sq * u + cq * side, sa * e[1] + ca * e[2] + p.d[i]])
        lw = -0.5 * (((np.array(m.p[:])[:, None] - e) / p.sigma_pos) ** 2).sum(0)
        return np.concatenate([q, qd]), lw - 0.5 * (((np.array(m.q[:])[:, None] - q) / p.sigma_enc) ** 2).sum(0)
    if model == "robotarm5":
        zp, za = z[:4], z[4:]
        q = s[:5] + dt * np.array(c.angles[:])[:, None] + np.float64(np.float32(0.2)) * za
        x, y = s[5] + s[7] * dt + np.float64(np.float32(0.2)) * zp[0], s[6] + s[8] * dt + np.float64(np.float32(0.2)) * zp[1]
        X, Y, _ = _arm_camera_point(q.T, x, y)
        lw = -0.1 * (((q - np.array(m.angles[:])[:, None]) ** 2).sum(0) + (X - m.x) ** 2 + (Y - m.y) ** 2)
        return np.concatenate([q, np.stack([x, y, s[7] + 2.0 * zp[2], s[8] + 2.0 * zp[3]])]), lw
    return None


def exact(case, seed):
    """The first step's posterior mean and weights.  Which particles live on after it depends on the last bit of 32-bit
    prefix sums, so nothing later has a value that more bits would settle; of a batch or a served track no estimate of
    the first step alone is read."""
    if case["kind"] != "filter" or case["model"] == "robotarm5_camera" or case["carry"]:
        return None
    params, ctrl, meas, dt, start, spread = _trace(case["model"], case["landmarks"], seed)
    n, V = case["m"] * case["G"], ea.NOISE_DIM[MODELS[case["model"]]]
    uniforms = (2 * case["m"] + 1 if case["resampler"] == "alias" else case["m"] + 1) * case["G"]
    size = -(-(V * n + uniforms) // (768 * 96)) * 768
    z = _normals(_mtgp_words(seed % 1000003, 96, size), n, V)
    s, lw = _weigh(case["model"], _start(case, seed, start, spread).astype(np.float64), z, params, ctrl[0], meas[0],
                   float(np.float32(dt)))
    log = case["weights"] == "log"
    w = np.exp(lw - lw.max()) if log else np.exp(lw)
    first = {"mean": (s * w).sum(1)[None] / w.sum(), "best": None, "weight": None, "block": None}
    later = {"mean": None, "best": None, "weight": None, "block": None}
    return {"first": first, "later": later, "particles": None, "weights": None}
