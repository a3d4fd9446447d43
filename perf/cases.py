"""The calls this framework is used for, with the sizes they are used at.

Each case names one way of calling the engine (`kind`) on one seeded graph:

  partition  Engine.partition() on a resident graph: merge phases, nodal
             sweeps and the search over the block count.  The default use,
             at the sizes of the N=1000, N=20000 and N=500000 workloads.
  drop_in    Graph_P(graph=...).partition(): the engine made, used and
             destroyed for one graph, as a program that partitions one graph
             after another does.
  resume     set_labels() + resume(): a known partition taken up again by
             the nodal chain.
  serve      serve.serve() of one graph whose edges arrive in increments.
  merge      one round of merge proposals on a state held by the engine.
  phase      restore() + merge proposals + carry-out: a merge phase as the
             search over the block count runs it.
  sweep      restore() + one nodal sweep over every node.
  mdl        set_labels() + degrees() + entropy(): the description length of
             a partition the caller has.

Graphs are directed degree-corrected block models from the package's seeded
generator; `weighted` ones carry weights 1..3, self-loops and a few nodes of
more than a thousand edges.  Every run() starts from what prepare() left and
gives the same outputs each time it is called.
"""
import math

import numpy as np

import usap_amd
from usap_amd import serve
from usap_amd._lib import lib


def _case(kind, N, K, B=0, dmax=100, p_in=0.7, init=0, ds_mode=0, batch=0, weighted=False,
          alpha=3.0, **more):
    """N nodes, K planted blocks, B blocks of the state (0: not used), nodal
    batches of `batch` nodes (0: the default, a quarter of the nodes)."""
    c = dict(kind=kind, N=N, K=K, B=B, dmax=dmax, p_in=p_in, init=init, ds_mode=ds_mode,
             batch=batch, weighted=weighted, alpha=alpha)
    c.update(more)
    return c


def listed():
    return [
        # the smallest graph people try first: a few hundred short launches
        _case("partition", 1000, 11, p_in=0.8, name="partition_1k"),
        # one graph after another, the engine's own making included
        _case("drop_in", 5000, 30, name="drop_in_5k"),
        # an ordinary graph with the defaults
        _case("partition", 20000, 32, p_in=0.6, alpha=0.8, name="partition_20k"),
        # weights, self-loops, hubs, the exact dS and one block per node to start
        _case("partition", 3001, 24, init=1, ds_mode=1, weighted=True,
              name="partition_weighted_3k"),
        # the largest: the headline workload
        _case("partition", 500000, 120, dmax=200, init=1, batch=4096, name="partition_500k"),
        # a known partition, taken up again after its graph has changed
        _case("resume", 50000, 76, name="resume_50k"),
        # one client's graph arriving in ten increments
        _case("serve", 20000, 53, stages=10, name="serve_20k"),
        # merge proposals in the middle of the search: few blocks, long rows
        _case("merge", 50000, 76, B=2500, name="merge_2500"),
        # a merge phase at the start of the search: many blocks, short rows
        _case("phase", 200000, 132, B=200000, name="phase_200k"),
        # one sweep after the first merge phase of a large graph
        _case("sweep", 200000, 132, B=100000, batch=4096, name="sweep_200k"),
        # scoring a partition: the smallest call and a large one
        _case("mdl", 1000, 11, B=11, p_in=0.8, name="mdl_1k"),
        _case("mdl", 200000, 132, B=132, name="mdl_200k"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["partition", "partition", "partition", "drop_in", "resume", "serve",
                       "merge", "phase", "sweep", "mdl"])
    hi = {"partition": 50000, "drop_in": 20000, "resume": 100000, "serve": 50000,
          "merge": 200000, "phase": 200000, "sweep": 200000, "mdl": 200000}[kind]
    N = _log_int(rng, 500, hi)
    # min_block 20 in the generator: K planted blocks need 20 K nodes
    K = max(2, int(round(N ** 0.4)))
    c = _case(kind, N, K, dmax=rng.choice([50, 100, 200]), p_in=round(rng.uniform(0.55, 0.85), 3),
              ds_mode=int(rng.random() < 0.25), weighted=rng.random() < 0.25)
    if kind in ("partition", "drop_in"):
        c["init"] = int(rng.random() < 0.3)
    if kind in ("merge", "phase", "sweep"):
        c["B"] = max(2, min(N, _log_int(rng, max(2, N // 500), N)))
    if kind == "mdl":
        c["B"] = max(1, min(N, _log_int(rng, 1, N)))
    if kind in ("sweep", "partition") and N >= 4096 and rng.random() < 0.5:
        c["batch"] = _log_int(rng, 1024, N)
    if kind == "serve":
        c["stages"] = rng.randint(2, 10)
    return c


def _graph(case, seed):
    g = usap_amd.generate_dcsbm(case["N"], case["K"], case["alpha"], 20, 10,
                                min(case["dmax"], case["N"] // 4), 2.5, case["p_in"], seed)
    if not case["weighted"]:
        return g
    rng = np.random.default_rng(seed + 1)
    N = g.N
    src, dst = g.edges()
    loops = rng.integers(0, N, max(1, N // 50))
    hubs = rng.integers(0, N, 4)
    fan = np.repeat(hubs, 600)
    ends = rng.integers(0, N, 2 * len(fan))
    src = np.concatenate([src, loops, fan, ends[len(fan):]])
    dst = np.concatenate([dst, loops, ends[:len(fan)], fan])
    perm = rng.permutation(len(src))
    w = rng.integers(1, 4, len(src))
    return usap_amd.Graph.from_edges(src[perm], dst[perm], N, w, g.truth)


def _params(case, seed):
    return dict(init=case["init"], ds_mode=case["ds_mode"], nodal_batch=case["batch"], seed=seed)


def _labels(case, g, seed):
    """Labels the caller has: B blocks (every one used) along the planted
    partition for `mdl`, the planted partition with a twentieth of the nodes
    elsewhere for `resume`."""
    rng = np.random.default_rng(seed + 2)
    if case["kind"] == "resume":
        lab = g.truth.copy()
        out = rng.random(g.N) < 0.05
        lab[out] = rng.integers(0, case["K"], int(out.sum()))
        return lab, case["K"]
    B = case["B"]
    order = np.lexsort((rng.random(g.N), g.truth))
    lab = np.empty(g.N, np.int32)
    lab[order] = (np.arange(g.N, dtype=np.int64) * B // g.N).astype(np.int32)
    if B == case["K"]:
        lab = g.truth.copy()
    return lab, B


def _merged(eng, case):
    """The state at B blocks, reached from one block per node by halving."""
    eng.set_labels(np.arange(case["N"], dtype=np.int32), case["N"])
    stream = 0
    while eng.B > case["B"]:
        _propose(eng, stream, None, None)
        eng.merge_apply(eng.B - max(case["B"], eng.B // 2))
        stream += 1
    eng.snapshot(0)


def _propose(eng, stream, s, dS):
    eng._ck(lib().usap_merge_propose(eng.h, eng.params.K, stream,
                                     None if s is None else s.ctypes.data,
                                     None if dS is None else dS.ctypes.data))


def prepare(case, seed):
    g = _graph(case, seed)
    kind, state = case["kind"], dict(case=case, graph=g, params=_params(case, seed))
    if kind == "drop_in":
        return state
    if kind == "serve":
        src, dst = g.edges()
        perm = np.random.default_rng(seed + 3).permutation(len(src))
        state["request"] = serve.ServedGraph(g.N, src[perm], dst[perm],
                                             w=None if g.out_w is None else g.out_w[perm])
        return state
    eng = state["engine"] = usap_amd.Engine(g, **state["params"])
    if kind in ("merge", "phase", "sweep"):
        _merged(eng, case)
    if kind in ("mdl", "resume"):
        state["labels"], state["B"] = _labels(case, g, seed)
    if kind in ("merge", "phase"):
        state["s"] = np.zeros(case["B"], np.int32)
        state["dS"] = np.zeros(case["B"], np.float64)
    return state


def _padded(values, dtype):
    """Per-phase values at a fixed length: the number of phases is an outcome."""
    out = np.zeros(64, dtype)
    out[:len(values)] = values
    return out


def run(state):
    case, eng = state["case"], state.get("engine")
    kind = case["kind"]
    if kind == "partition":
        labels, st = eng.partition()
        log = eng.partition_log()
        return dict(labels=labels, S=st["S"], B=st["B"], sweeps=st["sweeps"],
                    batches=st["batches"], moves=st["accepted_moves"],
                    phase_B=_padded([p["B"] for p in log], np.int64),
                    phase_S=_padded([p["S"] for p in log], np.float64),
                    phase_moves=_padded([p["moves"] for p in log], np.int64))
    if kind == "drop_in":
        p = usap_amd.Graph_P(graph=state["graph"])
        p.init, p.ds_mode, p.seed = case["init"], case["ds_mode"], state["params"]["seed"]
        labels = p.partition()
        return dict(labels=labels, S=p.stats["S"], B=p.stats["B"], sweeps=p.stats["sweeps"],
                    moves=p.stats["accepted_moves"])
    if kind == "resume":
        eng.set_labels(state["labels"], state["B"])
        labels, st = eng.resume(1 << 40)
        return dict(labels=labels, S=st["S"], sweeps=st["sweeps"], moves=st["accepted_moves"])
    if kind == "serve":
        labels, stages, _ = serve.serve([state["request"]], [0.0], state["params"],
                                        stages=case["stages"], workers=1,
                                        repartition_growth=2.0)
        rec = stages[0]
        return dict(labels=labels[0], S=np.array([r["S"] for r in rec], np.float64),
                    B=np.array([r["B"] for r in rec], np.int64),
                    sweeps=np.array([r["sweeps"] for r in rec], np.int64))
    if kind == "merge":
        _propose(eng, 100, state["s"], state["dS"])
        return dict(s=state["s"], dS=state["dS"])
    if kind == "phase":
        eng.restore(0)
        _propose(eng, 100, state["s"], state["dS"])
        eng.merge_apply(case["B"] // 2)
        do, di = eng.degrees()
        return dict(s=state["s"], dS=state["dS"], labels=eng.labels(), d_out=do, d_in=di)
    if kind == "sweep":
        eng.restore(0)
        sw = eng.nodal_sweep(case["batch"] or max(1, case["N"] // 4), 0, 0.0, 0.0, 1e-4, 0)
        do, di = eng.degrees()
        return dict(labels=eng.labels(), d_out=do, d_in=di, moves=sw["moves"],
                    dS=sw["dS_sum"], batches=sw["batches"])
    eng.set_labels(state["labels"], state["B"])
    do, di = eng.degrees()
    return dict(d_out=do, d_in=di, S=eng.entropy()[1])


def work(case):
    """Bytes that have to move, each list entry, label and result once per
    pass over the graph; there is no floating-point work to speak of.  A
    pass over the graph reads the list offsets and both lists (and weights)
    and the label at the other end of each entry."""
    N, B = case["N"], case["B"]
    E = 10 * N * (1.0 + 2.0 / (2.5 - 1.0))  # mean out-degree of d^-2.5 from 10 up, cut off
    entry = 8 if case["weighted"] else 4
    whole = 16 * N + 2 * E * (entry + 4) + 4 * N
    build = 16 * N + E * (2 * entry + 8) + 4 * N
    per = {
        # three phases at least (the search ends on a bracket of three block
        # counts), each with a build and two whole sweeps before its first test
        "partition": 3 * (build + 2 * whole) + 4 * N,
        "drop_in": 3 * (build + 2 * whole) + 4 * N + 2 * E * entry,
        "resume": build + 2 * whole + 4 * N,
        "serve": 3 * (build + 2 * whole) + 4 * N + 2 * E * entry,
        # every non-zero of M read once (at most one per edge), the result written
        "merge": min(E, B * B) * 12 + 24 * B,
        "phase": 2 * build + min(E, B * B) * 12 + 24 * B + 4 * N,
        "sweep": build + whole + 4 * N + 8 * B,
        "mdl": build + 8 * B,
    }[case["kind"]]
    return {"bytes": float(per), "flops": 0.0}


def exact(case, seed):
    """`mdl` has a closed form; every other result follows a random chain."""
    if case["kind"] != "mdl":
        return None
    g = _graph(case, seed)
    lab, B = _labels(case, g, seed)
    src, dst = g.edges()
    w = np.ones(g.E, np.float64) if g.out_w is None else g.out_w.astype(np.float64)
    a, b = lab[src].astype(np.int64), lab[dst].astype(np.int64)
    key, inv = np.unique(a * B + b, return_inverse=True)
    M = np.bincount(inv, weights=w, minlength=len(key))
    d_out = np.bincount(a, weights=w, minlength=B)
    d_in = np.bincount(b, weights=w, minlength=B)

    def xlogx(v):
        v = v[v > 0]
        return math.fsum(v * np.log(v))

    x = B * B / g.E
    model = g.E * (1 + x) * math.log(1 + x) - x * math.log(x) + g.N * math.log(B)
    data = xlogx(d_out) + xlogx(d_in) - xlogx(M)
    return dict(d_out=d_out.astype(np.int32), d_in=d_in.astype(np.int32), S=model + data)
