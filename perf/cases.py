"""Performance cases: the work that programs built on this framework have it do.

A case names one call (or one short sequence of calls) through the public entry points, on inputs
of the kind that call meets: leaf batches of searches, the playout batches of the drivers and of
bench.py, the labelling and training of the value network.  Every case is run as its caller runs
it -- results of host calls land in host memory, as the search that asked for them reads them
there; the allocation-free call leaves them in device memory.

    listed()        the named cases
    draw(rng)       one more case of the same ranges
    prepare, run    the inputs and handles a program holds, and one pass over them
    work(case)      bytes and operations one pass cannot do without
    exact(case, s)  the float outputs in 64 bits (network cases; playouts give whole numbers)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gpu_ai_amd import engine as ge

RANDOM, HEURISTIC, NOISY = ge.POLICY_RANDOM, ge.POLICY_HEURISTIC, ge.POLICY_HEURISTIC_NOISY

# Mean plies of a playout by policy, from openings (random) and midgames (the heuristics; positions
# up to 150 plies deep have about 35 left), and the int32 operations priced per ply: the frozen
# cost model of bench.py.
PLIES = {RANDOM: 53, HEURISTIC: 52, NOISY: 52}
OPS_PER_PLY = 192
# Multiply-adds of the 128-256-256-1 network per position: forward, and forward with the gradients
# of every parameter.
FWD_MADDS = 128 * 256 + 256 * 256 + 256
STEP_MADDS = FWD_MADDS + 128 * 256 + 2 * 256 * 256 + 2 * 256
PARAMS = ge.MLP_PARAMS


def listed():
    return [
        # One search's iteration: 256 leaves, one playout each, host buffers in and out.  The
        # smallest call of the framework, made thousands of times a move.
        dict(name="leaves-256", op="host", policy=RANDOM, n=256, per_pos=1, uneven=False,
             kmin=0, kmax=30, reject=False),
        # A batch iteration of one MCTS player with the reference's heuristic driver: some two
        # thousand distinct leaves, uneven trial counts.
        dict(name="mcts-noisy-2048x2", op="host", policy=NOISY, n=2048, per_pos=2, uneven=True,
             kmin=0, kmax=60, reject=False),
        # One iteration of 256 searches sharing the device: a graph replay of about 64k keyed
        # leaves, most of them distinct.
        dict(name="graph-21000x3", op="graph", policy=RANDOM, n=21000, per_pos=3, uneven=True,
             kmin=0, kmax=60, reject=False),
        # The host path's own size (bench.py's small workload).
        dict(name="random-64x4096", op="host", policy=RANDOM, n=64, per_pos=4096, uneven=False,
             kmin=0, kmax=30, reject=False),
        # The headline workload: a staged batch, launched and its winners fetched.
        dict(name="random-1024x1024", op="staged", policy=RANDOM, n=1024, per_pos=1024,
             uneven=False, kmin=0, kmax=30, reject=False),
        # The argmax heuristic on midgame positions, device buffers in and out without allocation.
        dict(name="noalloc-heuristic-1024x1024", op="noalloc", policy=HEURISTIC, n=1024,
             per_pos=1024, uneven=False, kmin=20, kmax=60, reject=True),
        # The reference's heuristic (noisy weights), host buffers, a count that is no power of two.
        dict(name="noisy-1000x999", op="host", policy=NOISY, n=1000, per_pos=999, uneven=False,
             kmin=20, kmax=60, reject=True),
        # Labelling for the value network: 256 playouts of every position, tallied on the device.
        dict(name="labels-65536x256", op="tally", policy=RANDOM, n=65536, per_pos=256,
             uneven=False, kmin=0, kmax=150, reject=True),
        # The positions of that labelling.
        dict(name="starts-262144", op="starts", n=262144, kmin=0, kmax=150, reject=True),
        # The network player's leaves of one iteration (4096 less the finished games among them).
        dict(name="net-forward-3900", op="forward", n=3900),
        # One batch's gradients from host buffers.
        dict(name="net-gradients-4096", op="gradients", n=4096),
        # One training epoch over a resident set, as a program that keeps the best weights runs it.
        dict(name="net-epoch-262144", op="epoch", n=262144, batch=4096),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["host", "host", "host", "graph", "staged", "noalloc", "tally", "starts",
                     "forward", "gradients", "epoch"])
    if op == "forward" or op == "gradients":
        return dict(op=op, n=_log(rng, 1, 4096))
    if op == "epoch":
        batch = 64 * _log(rng, 4, 64)
        return dict(op=op, n=_log(rng, 2 * batch, 262144), batch=batch)
    if op == "starts":
        kmax = rng.randint(10, 150)
        return dict(op=op, n=_log(rng, 64, 262144), kmin=rng.randint(0, min(kmax, 40)), kmax=kmax,
                    reject=rng.random() < 0.7)
    policy = rng.choice([RANDOM, RANDOM, HEURISTIC, NOISY])
    if op == "graph":  # search leaves: many positions, few playouts each
        n, per_pos, uneven = _log(rng, 200, 40000), rng.randint(1, 4), True
    elif op == "tally":
        n, per_pos, uneven = _log(rng, 256, 32768), _log(rng, 16, 512), rng.random() < 0.3
    elif op == "host" and rng.random() < 0.5:  # an MCTS iteration
        n, per_pos, uneven = _log(rng, 32, 16384), rng.randint(1, 3), rng.random() < 0.6
    else:  # a driver's batch
        n, per_pos, uneven = _log(rng, 16, 2048), _log(rng, 16, 1024), rng.random() < 0.4
    opening = rng.random() < 0.5
    return dict(op=op, policy=policy, n=n, per_pos=per_pos, uneven=uneven,
                kmin=0 if opening else 20, kmax=rng.choice([30, 60]) if opening else 60,
                reject=not opening)


# -- inputs -------------------------------------------------------------------------------------

_kept = {}


def _engine():
    """The program's device context (one per process, as a player or a trainer keeps it)."""
    if "engine" not in _kept:
        _kept["engine"] = ge.Engine(0)
    return _kept["engine"]


def _stream():
    """The stream of the calls that take device buffers."""
    if "stream" not in _kept:
        _kept["stream"] = torch.cuda.Stream()
    return _kept["stream"]


def _counts(case, rng):
    """Playouts per position: the trial counts of a batch are uneven, some positions get none (the
    total is the same for every seed)."""
    if not case["uneven"]:
        return None
    c = np.arange(case["n"], dtype=np.uint32)[::-1] % (2 * case["per_pos"] + 1)
    return rng.permutation(c.astype(np.uint32))


def _net_inputs(case, seed):
    """Positions (random placements of men and kings), targets and parameters of a network case,
    from the seed alone."""
    rng = np.random.default_rng([seed, case["n"]])
    n = case["n"]
    pos = np.zeros(n, dtype=ge.POS_DTYPE)
    squares = np.argsort(rng.random((n, 32)), axis=1).astype(np.uint32)
    a, b = rng.integers(1, 13, n), rng.integers(1, 13, n)
    at = np.arange(32)[None, :]
    bits = np.left_shift(np.uint32(1), squares)
    pos["p1"] = np.where(at < a[:, None], bits, 0).sum(1, dtype=np.uint32)
    pos["p2"] = np.where((at >= a[:, None]) & (at < (a + b)[:, None]), bits, 0).sum(1, dtype=np.uint32)
    crowned = np.where(rng.random((n, 32)) < rng.random((n, 1)) * 0.5, bits, 0).sum(1, dtype=np.uint32)
    pos["kings"] = crowned & (pos["p1"] | pos["p2"])
    pos["turn"] = rng.integers(0, 2, n)
    lead = (a - b) * np.where(pos["turn"] == 0, 1, -1)
    # labels of 256 playouts: the better side mostly wins
    win = rng.binomial(256, 1.0 / (1.0 + np.exp(-0.8 * lead)))
    t = ((2.0 * win - 256.0) / 256.0).astype(np.float32)
    w = np.zeros(PARAMS, np.float32)
    for lo, hi, fan in ((0, 32768, 128), (33024, 98560, 256), (98816, 99072, 256)):
        w[lo:hi] = rng.uniform(-1.0, 1.0, hi - lo) * math.sqrt(6.0 / fan)
    for lo, hi in ((32768, 33024), (98560, 98816), (99072, 99073)):
        w[lo:hi] = rng.uniform(-0.05, 0.05, hi - lo)
    return pos, t, w


def prepare(case, seed):
    op = case["op"]
    eng = _engine()
    s = {"case": case, "eng": eng, "seed": seed & 0xFFFFFFFF}
    if op == "starts":
        return s
    if op in ("forward", "gradients", "epoch"):
        pos, t, w = _net_inputs(case, seed)
        net = ge.ValueNet(eng, case.get("batch", 4096), seed=1)
        net.set_params(w)
        if op == "epoch":
            net.set_dataset(pos, t)
        s.update(net=net, pos=pos, t=t)
        return s
    rng = np.random.default_rng([seed, case["n"], case["per_pos"]])
    pos = eng.start_positions(s["seed"], case["n"], case["kmin"], case["kmax"], case["reject"])
    counts = _counts(case, rng)
    s.update(pos=pos, counts=counts, per_pos=None if counts is not None else case["per_pos"])
    if op == "graph":  # stream keys as the multi-search makes them: search << 16 | leaf
        leaf = np.arange(case["n"], dtype=np.uint32)
        s["keys"] = ((leaf // 256) << 16) | (leaf % 256)
        s["graph"] = eng.graph(case["n"], int(counts.sum()), case["policy"])
    elif op == "staged":
        s["eng"] = ge.Engine(0)
        s["eng"].stage(pos, per_pos=s["per_pos"], counts=counts)
    elif op == "noalloc":
        total = case["n"] * case["per_pos"] if counts is None else int(counts.sum())
        s["d_pos"] = torch.from_numpy(pos.view(np.uint8).copy()).cuda()
        s["d_counts"] = None if counts is None else torch.from_numpy(counts.view(np.int32)).cuda()
        s["d_winners"] = torch.zeros(total, dtype=torch.int8, device="cuda")
        s["d_status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["stream"] = _stream()
    return s


# -- one pass -----------------------------------------------------------------------------------

def _tallied(stats):
    return [stats["playouts"], stats["plies"], stats["max_moves"]]


def run(s):
    case, eng = s["case"], s["eng"]
    op = case["op"]
    if op == "host":
        r = eng.run_playouts(s["pos"], per_pos=s["per_pos"], counts=s["counts"], seed=s["seed"],
                             epoch=1, policy=case["policy"])
        return {"winners": r.winners, "stats": _tallied(r.stats)}
    if op == "graph":
        r = s["graph"].run(s["pos"], s["counts"], seed=s["seed"], epoch=1, keys=s["keys"])
        return {"winners": r.winners, "stats": _tallied(r.stats)}
    if op == "staged":
        st = eng.launch_staged(seed=s["seed"], epoch=1, policy=case["policy"])
        return {"winners": eng.fetch_winners(), "stats": _tallied(st)}
    if op == "tally":
        t, st = eng.run_tally(s["pos"], per_pos=s["per_pos"], counts=s["counts"], seed=s["seed"],
                              epoch=1, policy=case["policy"])
        return {"tallies": t.view(np.int32), "stats": _tallied(st)}
    if op == "noalloc":
        eng.run_playouts_noalloc(s["d_pos"].data_ptr(), case["n"],
                                 None if s["d_counts"] is None else s["d_counts"].data_ptr(),
                                 0 if s["per_pos"] is None else s["per_pos"],
                                 s["d_winners"].data_ptr(), seed=s["seed"], epoch=1,
                                 policy=case["policy"], d_status=s["d_status"].data_ptr(),
                                 stream=s["stream"].cuda_stream)
        return {"winners": s["d_winners"], "status": s["d_status"]}
    if op == "starts":
        p = eng.start_positions(s["seed"], case["n"], case["kmin"], case["kmax"], case["reject"])
        return {"positions": p.view(np.int32)}
    net = s["net"]
    if op == "forward":
        return {"values": net.forward(s["pos"])}
    if op == "gradients":
        g, loss = net.gradients(s["pos"], s["t"])
        return {"gradients": g, "loss": loss}
    loss, _ = net.train_epoch(case["batch"], 1e-3, s["seed"], 1)
    m, v, step = net.adam_state()
    return {"loss": loss, "params": net.get_params(), "m": m, "v": v, "step": step}


# -- what a pass cannot do without --------------------------------------------------------------

def work(case):
    op, n = case["op"], case["n"]
    if op == "forward":
        return {"bytes": 20 * n + 4 * PARAMS, "flops": 2 * FWD_MADDS * n}
    if op == "gradients":
        return {"bytes": 20 * n + 8 * PARAMS, "flops": 2 * STEP_MADDS * n}
    if op == "epoch":
        return {"bytes": 24 * n + 24 * PARAMS, "flops": 2 * STEP_MADDS * (n // case["batch"]) * case["batch"]}
    if op == "starts":  # random plies from the initial position; redrawn where the game is over
        return {"bytes": 16 * n, "flops": OPS_PER_PLY * n * (case["kmin"] + case["kmax"]) // 2}
    total = n * case["per_pos"]
    out = 12 * n if op == "tally" else total
    plies = PLIES[case["policy"]] if case["kmax"] <= 60 else 35
    return {"bytes": (24 if case["uneven"] else 16) * n + out,
            "flops": OPS_PER_PLY * plies * total}


# -- the network in 64 bits ---------------------------------------------------------------------

def _philox(c0, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (c0, 0, 3, c3), keys (k0, k1); c0 an array.
    Returns the words in order."""
    m32 = np.uint64(0xFFFFFFFF)
    x = [c0.astype(np.uint64), np.zeros_like(c0, np.uint64), np.full_like(c0, 3, np.uint64),
         np.full_like(c0, c3, np.uint64)]
    for r in range(10):
        a, b = x[0] * np.uint64(0xD2511F53), x[2] * np.uint64(0xCD9E8D57)
        ka, kb = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF), np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        x = [(b >> np.uint64(32)) ^ x[1] ^ ka, b & m32, (a >> np.uint64(32)) ^ x[3] ^ kb, a & m32]
    return np.stack(x, axis=1).reshape(-1)


def _epoch_order(n, seed, epoch):
    """The epoch's order: a Fisher-Yates shuffle whose swaps are drawn from the Philox words."""
    words = _philox(np.arange((n + 2) // 4 + 1, dtype=np.uint64), 1, seed, epoch)[:n - 1]
    swaps = (words % np.arange(n, 1, -1, dtype=np.uint64)).tolist()
    p = list(range(n))
    for c, j in enumerate(swaps):
        i = n - 1 - c
        p[i], p[j] = p[j], p[i]
    return np.array(p)


def _planes(pos):
    """The network's 128 inputs: own men, own kings, the opponent's men and kings, seen from the
    side to move (player 2's board rotated by 180 degrees)."""
    sq = np.arange(32, dtype=np.uint32)
    on = lambda m: ((m[:, None] >> sq) & 1).astype(bool)  # noqa: E731
    p1, p2, k = on(pos["p1"]), on(pos["p2"]), on(pos["kings"])
    second = (pos["turn"] != 0)[:, None]
    own = np.where(second, p2[:, ::-1], p1)
    opp = np.where(second, p1[:, ::-1], p2)
    k = np.where(second, k[:, ::-1], k)
    return torch.from_numpy(np.concatenate([own & ~k, own & k, opp & ~k, opp & k], 1)).double()


def _split(w):
    return [w[:32768].reshape(128, 256), w[32768:33024], w[33024:98560].reshape(256, 256),
            w[98560:98816], w[98816:99072], w[99072:]]


def _gradients(w, x, t):
    w = w.clone().requires_grad_()
    loss = ((_value(w, x) - t) ** 2).mean()
    return torch.autograd.grad(loss, w)[0], loss.detach()


def _value(w, x):
    w1, b1, w2, b2, w3, b3 = _split(w)
    h = torch.relu(torch.relu(x @ w1 + b1) @ w2 + b2)
    return torch.tanh(h @ w3 + b3)


def exact(case, seed):
    op = case["op"]
    if op not in ("forward", "gradients", "epoch"):
        return None
    pos, t, w = _net_inputs(case, seed)
    x, t, w = _planes(pos), torch.from_numpy(t).double(), torch.from_numpy(w).double()
    if op == "forward":
        return {"values": _value(w, x)}
    if op == "gradients":
        g, loss = _gradients(w, x, t)
        return {"gradients": g, "loss": float(loss)}
    batch = case["batch"]
    order = torch.from_numpy(_epoch_order(case["n"], seed & 0xFFFFFFFF, 1))
    m, v, total, steps = torch.zeros_like(w), torch.zeros_like(w), 0.0, case["n"] // batch
    for k in range(steps):
        rows = order[k * batch:(k + 1) * batch]
        g, loss = _gradients(w, x[rows], t[rows])
        total += float(loss)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return {"loss": total / steps, "params": w, "m": m, "v": v, "step": None}
