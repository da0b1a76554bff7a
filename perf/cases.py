"""The workloads whose speed this library is judged by: block Gibbs sampling
through the public Python API, over the range of models that it serves.

A case names a model family, its sizes, the chains and a schedule; `prepare`
builds what a user's program holds before the call (the model's arrays, the
compiled program, the chains on the device, the observer) and `run` makes one
call (or, for training, one step: new programs, initial states, gradients).
The families:

  lattice   Ising model on the L x L torus (sides that are a multiple of 32
            and sides that are not)
  er        Ising model on an Erdos-Renyi graph, greedy-coloured blocks
  potts     categorical model on the torus or on an Erdos-Renyi graph
  rbm       dense bipartite model, bf16 or f32 weights
  factors   spins and categorical nodes coupled by general discrete factors
  score     energies of a batch of given configurations
  grid_train, rbm_train
            one contrastive training step (IsingTrainingSpec,
            estimate_kl_grad, gradient ascent) of the sparse double grid and
            of the dense bipartite model

and what a pass returns (`op`): every observation's states on the host
("states"), the final states on the host ("run"), int64 moment sums in device
tensors ("moments"), moments through estimate_moments ("estimate").
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "thrml-rs_amd"))
import thrml_hip as th  # noqa: E402


def listed():
    return [
        # the first program a new user writes: one chain of a 10 x 10 torus,
        # every observation read back (hundreds of tiny half-sweeps)
        dict(name="lattice10_c1_states", family="lattice", op="states", L=10, C=1,
             warmup=10, samples=20, steps=2),
        # many chains of a small lattice for a long run, final states read back
        dict(name="lattice64_c256_run", family="lattice", op="run", L=64, C=256, sweeps=1000),
        # the headline configuration: large lattice, every node and edge
        # moment observed after every sweep, sums left on the device
        dict(name="lattice1024_c64_moments", family="lattice", op="moments", L=1024, C=64,
             warmup=1, samples=100, steps=1),
        # the large irregular graph: 1M nodes of mean degree 12
        dict(name="er1m_c32_moments", family="er", op="moments", N=1_000_000, degree=12.0, C=32,
             warmup=10, samples=10, steps=5),
        # a mid-size irregular graph with a ragged chain count, moments
        # through the one-call API (spec built per call, sums on the host)
        dict(name="er20k_c200_estimate", family="er", op="estimate", N=20011, degree=7.0, C=200,
             warmup=20, samples=20, steps=4),
        # labelling on a grid: 8 categories, final labels read back
        dict(name="potts512_q8_c32_run", family="potts", op="run", graph="torus", L=512, q=8,
             C=32, sweeps=100),
        # categorical model on an irregular graph, many categories, ragged chains
        dict(name="potts_er_q21_c50_run", family="potts", op="run", graph="er", N=10007,
             degree=8.0, q=21, C=50, sweeps=20),
        # the dense bipartite model on the matrix cores
        dict(name="rbm1024x4096_c4096_moments", family="rbm", op="moments", V=1024, H=4096,
             C=4096, f32=False, warmup=10, samples=10, steps=4),
        # one training step of the sparse double grid, one chain per phase, as
        # the reference trains it on images
        dict(name="grid40_c1_train", family="grid_train", side=40, visible=814, C=1, warmup=50,
             samples=10, steps=3),
        # one training step of a dense model with f32 weights
        dict(name="rbm512x1024_c256_train", family="rbm_train", V=512, H=1024, C=256, warmup=10,
             samples=10, steps=3),
        # spins and categorical nodes coupled by general factors
        dict(name="factors256_q4_c32_moments", family="factors", op="moments", L=256, q=4, C=32,
             warmup=10, samples=5, steps=5),
        # energies of a batch of configurations that arrive on the host
        dict(name="er100k_c128_score", family="score", graph="er", N=100_003, C=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges, no dearer than the largest listed one."""
    family = rng.choice(["lattice", "lattice", "er", "er", "potts", "potts", "rbm", "grid_train",
                         "rbm_train", "factors", "score"])
    c = dict(family=family)
    if family == "lattice":
        c.update(op=rng.choice(["states", "run", "moments", "estimate"]), L=_log_int(rng, 8, 1024))
        if rng.random() < 0.5:  # the sides of the threshold-table kernel
            c["L"] = max(32, c["L"] // 32 * 32)
        c["C"] = _log_int(rng, 1, max(1, min(1024, (64 << 20) // c["L"] ** 2)))
        n, per_node = c["L"] ** 2, 1.0
    elif family == "er":
        c.update(op=rng.choice(["states", "run", "moments", "estimate"]),
                 N=_log_int(rng, 100, 300_000), degree=round(rng.uniform(3.0, 14.0), 1))
        c["C"] = _log_int(rng, 1, max(1, min(1024, (32 << 20) // c["N"])))
        n, per_node = c["N"], 6.0
    elif family == "potts":
        c.update(op="run", graph=rng.choice(["torus", "er"]),
                 q=rng.choice([2, 3, 4, 5, 6, 8, 10, 12, 16, 21, 32, 48]))
        # at most 32M weights
        if c["graph"] == "torus":
            c["L"] = 2 * _log_int(rng, 6, min(256, int(2000 / c["q"])))
            n = c["L"] ** 2
        else:
            c["degree"] = round(rng.uniform(3.0, 12.0), 1)
            c["N"] = _log_int(rng, 100, min(60_000, int(64e6 / c["degree"] / c["q"] ** 2)))
            n = c["N"]
        c["C"] = _log_int(rng, 1, 128)
        per_node = 2.0 * c["q"]
    elif family in ("rbm", "rbm_train"):
        c.update(V=_log_int(rng, 64, 1024), H=_log_int(rng, 64, 2048))
        if family == "rbm":
            c.update(op=rng.choice(["run", "moments"]), f32=rng.random() < 0.5)
        c["C"] = _log_int(rng, 16, 4096 if family == "rbm" else 512)
        n, per_node = c["V"] + c["H"], 4.0
    elif family == "grid_train":
        c.update(side=rng.randrange(20, 61))
        c.update(visible=int(c["side"] ** 2 * rng.uniform(0.2, 0.6)), C=_log_int(rng, 1, 64))
        n, per_node = 2 * c["side"] ** 2, 4.0
    elif family == "factors":
        c.update(op=rng.choice(["run", "moments"]), L=2 * _log_int(rng, 8, 128),
                 q=rng.choice([2, 3, 4, 6, 8, 12]), C=_log_int(rng, 1, 64))
        n, per_node = 2 * c["L"] ** 2, 8.0
    else:
        c.update(graph=rng.choice(["torus", "er"]), N=_log_int(rng, 1000, 200_000),
                 C=_log_int(rng, 1, 256))
        return c
    # the sweeps of the pass, so that it stays below the largest listed one
    budget = max(4, min(400, int(4e9 / (per_node * n * max(c["C"], 16)))))
    sweeps = _log_int(rng, 4, max(4, budget))
    if c.get("op") == "run":
        c["sweeps"] = sweeps
    else:
        samples = max(2, min(20, sweeps // 2))
        if c.get("op") == "states":  # the observations' bytes on the host
            samples = max(2, min(samples, (32 << 20) // (n * c["C"])))
        c.update(warmup=max(1, sweeps // 3), samples=samples,
                 steps=max(1, (sweeps - sweeps // 3) // samples))
    return c


# ---------------------------------------------------------------------------
# models

_DEVICE = []


def _device():
    """The program's one library context, on torch's current stream."""
    if not _DEVICE:
        d = th.Device(0)
        d.set_stream(torch.cuda.current_stream().cuda_stream)
        _DEVICE.append(d)
    return _DEVICE[0]


@functools.lru_cache(maxsize=8)
def _torus(L):
    n, edges, up, lo = th.make_nearest_neighbor_lattice(L, True)
    return n, edges, (up, lo)


@functools.lru_cache(maxsize=8)
def _er(N, degree):
    edges = th.erdos_renyi(N, degree / (N - 1), 2003)
    return N, edges, tuple(th.coloring_to_blocks(th.greedy_coloring(N, edges)))


@functools.lru_cache(maxsize=4)
def _grid(side, visible):
    return th.double_grid(side, [1, 4, 15], visible, 0)


def _normal(gen, shape, mean, std):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return x.mul_(std).add_(mean).cpu().numpy()


def _bits(gen, shape, p=0.5):
    x = torch.rand(shape, generator=gen, device="cuda")
    return (x < p).to(torch.uint8).cpu().numpy()


def _graph(case):
    """(nodes, edges, blocks) of a lattice, er, potts or score case."""
    if case["family"] == "lattice" or case.get("graph") == "torus":
        return _torus(case["L"] if "L" in case else max(4, int(math.sqrt(case["N"]))))
    return _er(case["N"], case.get("degree", 8.0))


def _ising(case, gen):
    n, edges, blocks = _graph(case)
    lattice = case["family"] == "lattice" or case.get("graph") == "torus"
    b = _normal(gen, n, 0.0, 0.1 if lattice else 0.2)
    w = _normal(gen, edges.shape[0], 0.4 if lattice else 0.0, 0.05 if lattice else 0.3)
    return th.IsingEBM(n, edges, b, w, 1.0), list(blocks)


def _factors(case, gen):
    """A two-layer torus: spins S and q-state nodes X = S + n, spin biases and
    couplings, categorical biases and square pair factors, and one
    spin-categorical factor per site."""
    n, edges, (up, lo) = _torus(case["L"])
    q = case["q"]
    S = np.arange(n, dtype=np.uint32)
    X = S + np.uint32(n)
    eu, ev = edges[:, 0].astype(np.uint32), edges[:, 1].astype(np.uint32)
    E = eu.size
    fs = [th.SpinEBMFactor([S], _normal(gen, (n, 1, 1), 0.0, 0.2)),
          th.SpinEBMFactor([eu, ev], _normal(gen, (E, 1, 1), 0.3, 0.1)),
          th.CategoricalEBMFactor([X], _normal(gen, (n, q, 1), 0.0, 0.3)),
          th.SquareCategoricalEBMFactor([X[eu], X[ev]], _normal(gen, (E, q, q), 0.0, 0.3)),
          th.DiscreteEBMFactor([S], [X], _normal(gen, (n, q, 1), 0.0, 0.3))]
    kinds = np.concatenate([np.zeros(n, np.uint8), np.ones(n, np.uint8)])
    blocks = [up.nodes, lo.nodes, up.nodes + np.uint32(n), lo.nodes + np.uint32(n)]
    return 2 * n, kinds, fs, [th.Block(b) for b in blocks]


def _rbm_edges(V, H):
    v = np.repeat(np.arange(V, dtype=np.uint32), H)
    h = np.tile(np.arange(V, V + H, dtype=np.uint32), V)
    return np.stack([v, h], axis=1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dev, fam, C = _device(), case["family"], case["C"]
    s = dict(case=case, key=th.RngKey(seed + 1))
    k_init = th.RngKey(seed + 2)
    if fam in ("lattice", "er"):
        ebm, blocks = _ising(case, gen)
        s["prog"] = th.IsingSamplingProgram(ebm, blocks, [], dev)
        s["state"] = th.hinton_init(k_init, s["prog"], C)
        nodes, edges = np.arange(ebm.n_nodes, dtype=np.uint32), ebm.edges
    elif fam == "rbm":
        W = _normal(gen, (case["V"], case["H"]), 0.0, 0.05)
        if not case["f32"]:
            W = th.bf16_round(W)[0]
        bv = _normal(gen, case["V"], 0.0, 0.1)
        bh = _normal(gen, case["H"], 0.0, 0.1)
        s["prog"] = th.RbmProgram(W, bv, bh, 1.0, dev)
        s["state"] = th.hinton_init(k_init, s["prog"], C)
        nodes = np.arange(case["V"] + case["H"], dtype=np.uint32)
        # the moments of a few couplings besides every node's
        edges = np.stack([np.arange(64), case["V"] + np.arange(64)], axis=1)
    elif fam == "potts":
        n, edges, blocks = _graph(case)
        q = case["q"]
        W = _normal(gen, (edges.shape[0], q, q), 0.0, 0.2)
        bias = _normal(gen, (n, q), 0.0, 0.1)
        s["prog"] = th.CategoricalProgram(n, q, edges, W, bias, list(blocks), dev)
        s["state"] = s["prog"].new_state(C)
        x = torch.randint(0, q, (C, n), generator=gen, device="cuda", dtype=torch.uint8)
        s["state"].set_global(x.cpu().numpy())
    elif fam == "factors":
        n, kinds, fs, blocks = _factors(case, gen)
        s["prog"] = th.FactorSamplingProgram(kinds, case["q"], fs, blocks, [], dev)
        s["state"] = s["prog"].new_state(C)
        s["state"].set_global(_bits(gen, (C, n)))
        # first moments of every node of the sampled layers
        s["spec"] = [[[i] for i in range(n)]]
    elif fam == "score":
        ebm, blocks = _ising(case, gen)
        s["prog"] = th.IsingSamplingProgram(ebm, blocks, [], dev)
        s["state"] = s["prog"].new_state(C)
        s["x"] = _bits(gen, (C, ebm.n_nodes))
    else:
        if fam == "grid_train":
            up, lo, vis, rest, n, edges = _grid(case["side"], case["visible"])
            s["blocks"] = ([vis], [rest, lo], [up, lo])
        else:
            V, H = case["V"], case["H"]
            n, edges = V + H, _rbm_edges(V, H)
            vis, hid = th.Block(np.arange(V)), th.Block(np.arange(V, V + H))
            s["blocks"] = ([vis], [hid], [vis, hid])
        s["n"], s["edges"], s["dense"] = n, edges, fam == "rbm_train"
        s["nodes"] = np.arange(n, dtype=np.uint32)
        # a model some steps into its training, and a batch of data rows
        s["w"] = _normal(gen, edges.shape[0], 0.0, 0.02)
        s["b"] = _normal(gen, n, 0.0, 0.02)
        s["data"] = _bits(gen, (10, len(vis)), 0.3).astype(np.float32)
        s["dev"] = dev
    if "samples" in case:
        s["schedule"] = th.SamplingSchedule(case["warmup"], case["samples"], case["steps"])
    if case.get("op") == "moments":
        if fam == "factors":
            s["observer"] = th.MomentAccumulatorObserver(s["prog"], s["spec"])
        else:
            s["observer"] = th.MomentAccumulatorObserver(s["prog"],
                                                         th.ising_moment_spec(nodes, edges))
            s["out"] = (torch.zeros(nodes.size, dtype=torch.int64, device="cuda"),
                        torch.zeros(edges.shape[0], dtype=torch.int64, device="cuda"))
    elif case.get("op") == "estimate":
        s["nodes"], s["edges"] = nodes, edges
    return s


# ---------------------------------------------------------------------------
def _train_step(s):
    k_pos, k_neg, s["key"] = s["key"].split(3)
    data_blocks, pos_blocks, neg_blocks = s["blocks"]
    ebm = th.IsingEBM(s["n"], s["edges"], s["b"], s["w"], 1.0)
    spec = th.IsingTrainingSpec(ebm, data_blocks, [], pos_blocks, neg_blocks, s["schedule"],
                                s["schedule"], s["dev"], dense=s["dense"])
    C = s["case"]["C"]
    init_pos = th.hinton_init(k_pos, spec.program_positive, C)
    init_neg = th.hinton_init(k_neg, spec.program_negative, C)
    gw, gb = th.estimate_kl_grad(k_pos, spec, s["nodes"], s["edges"], [s["data"]], [], init_pos,
                                 init_neg)
    lr = np.float32(0.01)
    s["w"] = s["w"] + lr * gw
    s["b"] = s["b"] + lr * gb
    init_pos.close()
    init_neg.close()
    spec.close()
    return {"grad_w": gw, "grad_b": gb, "w": s["w"], "b": s["b"]}


def run(s):
    case = s["case"]
    if case["family"] == "score":
        s["state"].set_global(s["x"])
        return th.ising_energy(s["prog"], s["state"])
    if case["family"] in ("grid_train", "rbm_train"):
        return _train_step(s)
    key, s["key"] = s["key"].split_two()
    prog, state, op = s["prog"], s["state"], case["op"]
    if op == "states":
        return th.sample_states(key, prog, s["schedule"], state)
    if op == "moments":
        if "out" in s:
            return s["observer"].sample_with_observation(key, s["schedule"], state, out=s["out"])
        return s["observer"].sample_with_observation(key, s["schedule"], state)
    if op == "estimate":
        return th.estimate_moments(key, s["nodes"], s["edges"], prog, s["schedule"], state,
                                   return_sums=True)
    th.run_blocks(key, prog, state, (), case["sweeps"])
    return state.get_global()


# ---------------------------------------------------------------------------
def _sizes(case):
    """(nodes, edges, floats of parameters, arithmetic per node update) of a
    case; an update takes one keystream word (a 16th of a ChaCha8 block's
    about 360 operations) per spin, or one per category, its neighbour sum
    and its decision."""
    fam = case["family"]
    word, decide = 23, 8
    if fam in ("lattice", "er", "score"):
        n, edges, _ = _graph(case)
        E = edges.shape[0]
        return n, E, n + E, 2.0 * 2 * E / n + word + decide
    if fam == "potts":
        n, edges, _ = _graph(case)
        E, q = edges.shape[0], case["q"]
        return n, E, n * q + E * q * q, q * (2.0 * E / n + word + decide)
    if fam in ("rbm", "rbm_train"):
        V, H = case["V"], case["H"]
        return V + H, V * H, V + H + V * H, 4.0 * V * H / (V + H) + word + decide
    if fam == "factors":
        n, edges, _ = _torus(case["L"])
        E, q = edges.shape[0], case["q"]
        per = (2.0 * 2 * E / n + 2 + word + decide) + q * (2.0 * E / n + 2 + word + decide)
        return 2 * n, 2 * E, n + E + 2 * n * q + E * q * q, per / 2
    n, edges = _grid(case["side"], case["visible"])[4:6]
    E = edges.shape[0]
    return n, E, n + E, 2.0 * 2 * E / n + word + decide


def _sweeps(case):
    if "sweeps" in case:
        return case["sweeps"]
    return case["warmup"] + (case["samples"] - 1) * case["steps"]


def work(case):
    n, E, params, per = _sizes(case)
    C = case["C"]
    state = C * n / 8.0 if case["family"] in ("lattice", "er", "rbm") else float(C * n)
    if case["family"] == "score":
        return {"bytes": 4.0 * params + 8 * E + C * n + 8 * C, "flops": 2.0 * C * (n + E)}
    if case["family"] in ("grid_train", "rbm_train"):
        # two phases; gradients and updated weights out
        return {"bytes": 4.0 * params + 8.0 * E + 16.0 * (n + E),
                "flops": 2.0 * _sweeps(case) * C * n * per}
    out = {"run": float(C * n), "states": float(case.get("samples", 0) * C * n),
           "moments": 8.0 * (n + (E if case["family"] in ("lattice", "er") else 0)),
           "estimate": 8.0 * (n + E)}[case["op"]]
    indices = 0 if case["family"] == "lattice" or case.get("graph") == "torus" else 8 * E
    return {"bytes": 4.0 * params + indices + 2 * state + out,
            "flops": float(_sweeps(case)) * C * n * per}


def tolerance(case):
    # energies are 64-bit sums of 32-bit terms: another order of the sum moves
    # them by about 2e-16 of the terms' root sum of squares.  Everything else
    # is a count, a category or a quotient of counts, and the streams of
    # uniforms are fixed by the key.
    if case["family"] == "score":
        return {"rel": 1e-12, "max": 1e-11}
    return "exact"


def exact(case, seed):
    """The energies of the given configurations in 64 bits; the sampled
    outputs are whole numbers (or quotients of them) and have no such value."""
    if case["family"] != "score":
        return None
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ebm, blocks = _ising(case, gen)
    x = _bits(gen, (case["C"], ebm.n_nodes))
    order = np.concatenate([b.nodes for b in blocks])
    s = torch.empty(x.shape, dtype=torch.float64, device="cuda")
    s[:, torch.from_numpy(order.astype(np.int64))] = torch.from_numpy(x).cuda().double() * 2 - 1
    u = torch.from_numpy(ebm.edge_u.astype(np.int64)).cuda()
    v = torch.from_numpy(ebm.edge_v.astype(np.int64)).cuda()
    b = torch.from_numpy(ebm.biases).cuda().double()
    w = torch.from_numpy(ebm.weights).cuda().double()
    e = torch.empty(case["C"], dtype=torch.float64, device="cuda")
    for c in range(case["C"]):
        e[c] = -ebm.beta * ((b * s[c]).sum() + (w * s[c, u] * s[c, v]).sum())
    return e.cpu().numpy()
