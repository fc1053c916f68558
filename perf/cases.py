"""The work that users of this library have it do, as cases that can be timed.

A case is a dict of plain values; its "kind" says which entry points it goes
through:

  pipeline  the class mirror from the model on: table, SCCs and order, one FP64
            solve on host arrays (what every program written against the
            reference's classes does per model);
  plan      one batch of rate sets on a plan that the program keeps
            (solve_plan.solve), device arrays in and out;
  many      batches of several networks in one call (solve_plan.solve_many);
  forward   the surrogate's probabilities for a batch of rate sets;
  train     one run of Adam steps of the surrogate, and its parameters after.

Networks come from paraexastolog_amd.synth by family (c1: N nodes reading 2 or
3 others, 5 fixed nodes; c2: 2 inputs, no fixed node; c3: 3 inputs and three
spliced 3-cycles, 5 fixed nodes), size and seed; the seed of a measurement draws
the rates, so another seed is another batch on the same network.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from paraexastolog_amd import (cu_context, initial_state, model_builder, solve_plan, solver, synth, transition_graph,
                               transition_rates, transition_table)
from paraexastolog_amd.surrogate import Surrogate

# Seeds of drawn networks.  Any seed gives a valid network; left out of c1 are four
# whose systems are so ill-conditioned at some size that single rate sets miss the
# tolerances below (the call then says so) or take many seconds.
SEEDS = {"c1": [s for s in range(24) if s not in (4, 6, 8, 19)], "c2": range(24), "c3": range(24)}
MLP_HIDDEN, MLP_LAYERS = 256, 3


def listed():
    return [
        # a toy-sized model through the whole class API: launches and host round trips are all of it
        {"name": "pipeline n10", "kind": "pipeline", "family": "c2", "N": 10, "net": 6},
        # a model of the size of the small published ones (13 to 15 nodes)
        {"name": "pipeline n15", "kind": "pipeline", "family": "c1", "N": 15, "net": 2},
        # a model of the size of the large published ones (20 nodes and more), the headline's network
        {"name": "pipeline n20", "kind": "pipeline", "family": "c1", "N": 20, "net": 0},
        # one rate set at a time in FP64 on a kept plan (a parameter study that steps set by set)
        {"name": "plan n20 one fp64", "kind": "plan", "family": "c1", "N": 20, "net": 0, "sets": 1, "precision": 0,
         "tol": 1e-13, "graph": 0},
        # the headline batch: 1024 sets of one N=20 network, mixed precision, replayed as a HIP graph
        {"name": "plan n20 1024", "kind": "plan", "family": "c1", "N": 20, "net": 0, "sets": 1024, "precision": 1,
         "tol": 1e-12, "graph": 1},
        # an odd-sized FP64 batch of a 2048-state terminal component
        {"name": "plan n16 250 fp64", "kind": "plan", "family": "c2", "N": 16, "net": 11, "sets": 250, "precision": 0,
         "tol": 1e-12, "graph": 0},
        # absorption into two attractors: 44,992 states undecided between them
        {"name": "plan n16 absorb 100", "kind": "plan", "family": "c2", "N": 16, "net": 0, "sets": 100, "precision": 1,
         "tol": 1e-12, "graph": 0},
        # half a million unknowns per set, few sets
        {"name": "plan n20 wide 16", "kind": "plan", "family": "c1", "N": 20, "net": 7, "sets": 16, "precision": 1,
         "tol": 1e-12, "graph": 0},
        # the mixed-precision network: a terminal component of 221,184 states, 64 sets
        {"name": "plan n22 64", "kind": "plan", "family": "c3", "N": 22, "net": 8, "sets": 64, "precision": 1,
         "tol": 1e-12, "graph": 0},
        # eight networks of uneven size in one call
        {"name": "many uneven 8x128", "kind": "many", "networks": 8, "net": 0, "sets": 128, "precision": 1,
         "tol": 1e-12, "graph": 0},
        # the learned warm start: prediction for a batch of rate sets
        {"name": "forward 4096", "kind": "forward", "rows": 4096, "n_in": 32, "n_out": 2048},
        # and its training, on minibatches of 512 rows
        {"name": "train 64x512", "kind": "train", "rows": 512, "steps": 64, "n_in": 32, "n_out": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        if case["kind"] in ("forward", "train") or any(_has_system(net) for net in _networks(case)):
            return case


def _draw(rng):
    kind = rng.choice(["pipeline", "pipeline", "plan", "plan", "plan", "plan", "many", "forward", "train"])
    if kind == "pipeline":
        family = rng.choice(["c1", "c2"])
        return {"kind": kind, "family": family, "N": rng.randint(8, 18) if family == "c1" else rng.randint(6, 17),
                "net": rng.choice(SEEDS[family])}
    if kind == "plan":
        family = rng.choice(["c1", "c1", "c2", "c2", "c3"])
        N = {"c1": rng.randint(10, 18), "c2": rng.randint(8, 17), "c3": rng.randint(16, 19)}[family]
        # the larger systems come in smaller batches, as their solves take hundreds of times longer
        most = 24 if family == "c3" else 1500 if N <= 12 else 200 if N <= 15 else 48
        return {"kind": kind, "family": family, "N": N, "net": rng.choice(SEEDS[family]),
                "sets": _log_int(rng, 1, most), "precision": rng.randrange(2), "tol": rng.choice([1e-12, 1e-11]),
                "graph": rng.randrange(2)}
    if kind == "many":
        return {"kind": kind, "networks": rng.randint(2, 5), "net": rng.randrange(24), "sets": rng.randint(1, 100),
                "precision": rng.randrange(2), "tol": 1e-12, "graph": 0}
    case = {"kind": kind, "n_in": 2 * rng.randint(6, 22), "n_out": _log_int(rng, 10, 2048)}
    if kind == "forward":
        return dict(case, rows=_log_int(rng, 1, 4096))
    return dict(case, rows=_log_int(rng, 16, 512), steps=rng.randint(1, 64))


# ---- networks ---------------------------------------------------------------

def _network(family, N, seed):
    if family == "c1":
        return synth.generate(N, 0, seed, 5)[0]
    if family == "c2":
        return synth.generate(N, 2, seed, 0)[0]
    net, rng = synth.generate(N, 3, seed, 5)
    synth.splice_cycles(net, rng, 3)
    return net


def _networks(case):
    if case["kind"] == "many":
        return [net for net, _ in synth.uneven(case["net"])][:case["networks"]]
    return [_network(case["family"], case["N"], case["net"])]


def _rates(case, seed):
    """One [sets][2N] array of log-uniform [0.1, 10] rates per network."""
    rng = np.random.default_rng(seed)
    sets = case.get("sets", 1)
    return [np.exp(rng.uniform(math.log(0.1), math.log(10.0), (sets, 2 * net.N))) for net in _networks(case)]


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = cu_context(0)
    return _ctx


def _ptr(t):
    return C.c_void_p(t.data_ptr())


class _Kept:
    """What a program keeps per network: model, table, graph, plan and its device arrays."""

    def __init__(self, net, rates):
        ctx = _context()
        self.model = model_builder().parse_model(net.bnet())
        self.table = transition_table(ctx, self.model, rates[0])
        self.table.construct_table()
        self.graph = transition_graph(ctx, self.table)
        self.graph.reorganize_vertices()
        fixed, vals = net.fixed_spec()
        x0 = torch.from_numpy(initial_state(self.model.nodes, fixed, vals).state).cuda()
        self.plan = solve_plan(ctx, self.table, _ptr(x0))
        self.rates = torch.from_numpy(rates).cuda()
        self.final = torch.empty((len(rates), 1 << net.N), dtype=torch.float64, device="cuda")


def _dims(case):
    return [case["n_in"]] + [MLP_HIDDEN] * MLP_LAYERS + [case["n_out"]]


def _mlp_inputs(case, seed):
    """Parameters (He initialisation), log-rates and targets (skewed distributions, as terminal vectors are)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    params = []
    for a, b in zip(_dims(case)[:-1], _dims(case)[1:]):
        params += [torch.randn((a, b), generator=g, device="cuda") * math.sqrt(2.0 / a),
                   torch.randn(b, generator=g, device="cuda") * 0.01]
    rows = case["rows"] * case.get("steps", 1)
    x = (torch.rand((rows, case["n_in"]), generator=g, device="cuda") * 2 - 1) * math.log(10.0)
    t = None
    if case["kind"] == "train":
        t = torch.softmax(3.0 * torch.randn((rows, case["n_out"]), generator=g, device="cuda"), 1)
    return params, x, t


LR_FIRST, LR_LAST = 3e-4, 1e-4  # the second half of surrogate.train's default decay


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pipeline":
        net = _networks(case)[0]
        model = model_builder().parse_model(net.bnet())
        rates = transition_rates(model)
        rates.rates = _rates(case, seed)[0][0]
        fixed, vals = net.fixed_spec()
        return {"case": case, "model": model, "rates": rates, "x0": initial_state(model.nodes, fixed, vals)}
    if kind in ("plan", "many"):
        kept = [_Kept(net, r) for net, r in zip(_networks(case), _rates(case, seed))]
        return {"case": case, "kept": kept,
                "opts": {k: case[k] for k in ("precision", "tol", "graph")}}
    params, x, t = _mlp_inputs(case, seed)
    sur = Surrogate(_context(), case["n_in"], case["n_out"], hidden=MLP_HIDDEN, hidden_layers=MLP_LAYERS)
    sur.set_params(torch.cat([p.reshape(-1) for p in params]).cpu().numpy())
    state = {"case": case, "sur": sur, "x": x, "t": t}
    if kind == "forward":
        state["probs"] = torch.empty((case["rows"], case["n_out"]), dtype=torch.float32, device="cuda")
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pipeline":
        ctx = _context()
        table = transition_table(ctx, state["model"], state["rates"].rates)
        table.construct_table()
        graph = transition_graph(ctx, table)
        graph.reorganize_vertices()
        s = solver(ctx, table, graph, state["rates"], state["x0"])
        s.solve()
        return {"final": s.final_state, "order": graph.reordered_vertices, "offsets": graph.sccs_offsets,
                "scc": graph.scc_ids, "terminals": graph.terminals_count}
    if kind == "plan":
        k = state["kept"][0]
        k.plan.solve(case["sets"], _ptr(k.rates), _ptr(k.final), **state["opts"])
        return {"final": [k.final]}
    if kind == "many":
        kept = state["kept"]
        solve_plan.solve_many(_context(), [k.plan for k in kept], [case["sets"]] * len(kept),
                              [_ptr(k.rates) for k in kept], [_ptr(k.final) for k in kept], **state["opts"])
        return {"final": [k.final for k in kept]}
    if kind == "forward":
        state["sur"].forward_device(case["rows"], _ptr(state["x"]), _ptr(state["probs"]))
        return {"probs": state["probs"]}
    loss = state["sur"].train_steps_device(case["steps"], case["rows"], _ptr(state["x"]), _ptr(state["t"]), LR_FIRST,
                                           LR_LAST)
    return {"loss": loss, "params": state["sur"].params()}


def work(case):
    """Inputs read once and outputs written once; for the surrogate also its products."""
    kind = case["kind"]
    if kind == "pipeline":
        # initial vector and final vector (FP64), order and component ids (int32)
        return {"bytes": 24.0 * (1 << case["N"]), "flops": 0.0}
    if kind in ("plan", "many"):
        return {"bytes": float(sum(8 * case["sets"] * ((1 << net.N) + 2 * net.N) for net in _networks(case))),
                "flops": 0.0}
    d = _dims(case)
    weights = sum(a * b + b for a, b in zip(d[:-1], d[1:]))
    rows = case["rows"] * case.get("steps", 1)
    if kind == "forward":
        return {"bytes": 4.0 * (weights + rows * (d[0] + d[-1])), "flops": 2.0 * rows * weights}
    # each step's inputs and targets are read; parameters come out once (three products per weight)
    return {"bytes": 4.0 * (2 * weights + rows * (d[0] + d[-1])), "flops": 6.0 * rows * weights}


# ---- the same results in 64 bits, by plain numpy and torch ------------------

def _flip_masks(net):
    """mask[s] bit i: the rule of node i differs from bit i of s."""
    s = np.arange(1 << net.N, dtype=np.int64)
    mask = np.zeros(1 << net.N, dtype=np.int64)
    for i in range(net.N):
        idx = np.zeros(1 << net.N, dtype=np.int64)
        for k, j in enumerate(net.inputs[i]):
            idx |= ((s >> j) & 1) << k
        mask |= (np.asarray(net.tables[i], dtype=np.int64)[idx] ^ ((s >> i) & 1)) << i
    return mask


def _closure(mask, N, seeds, forward):
    """States reachable from `seeds` (forward) or reaching them."""
    seen = np.zeros(1 << N, dtype=bool)
    seen[seeds] = True
    front = np.asarray(seeds, dtype=np.int64)
    while front.size:
        new = []
        for i in range(N):
            u = front ^ (1 << i)
            edge = (mask[front] if forward else mask[u]) >> i & 1
            u = u[(edge == 1) & ~seen[u]]
            seen[u] = True
            new.append(u)
        front = np.unique(np.concatenate(new))
    return seen


def _start(net):
    """Mask of the states that the initial distribution is uniform over."""
    s = np.arange(1 << net.N, dtype=np.int64)
    start = np.ones(1 << net.N, dtype=bool)
    for i, v in zip(net.fixed, net.fixed_vals):
        start &= (s >> i & 1) == v
    return start


def _has_system(net):
    """Whether the final vector depends on the rates: a reachable attractor of several states, or a choice of two."""
    mask = _flip_masks(net)
    reach = _closure(mask, net.N, np.flatnonzero(_start(net)), True)
    parts = _terminal_components(mask, net.N, reach)
    return any(len(states) > 1 for states, _ in parts) or bool((np.sum([b for _, b in parts], axis=0) > 1).any())


def _terminal_components(mask, N, reach):
    """Terminal components among the `reach` states, each with the states that reach it."""
    rng = np.random.default_rng(0)
    left, found = reach.copy(), []
    while left.any():
        s = int(np.flatnonzero(left)[0])
        while True:
            for _ in range(4 * (1 << min(N, 12))):  # a random walk ends up in a terminal component
                bits = [i for i in range(N) if mask[s] >> i & 1]
                if not bits:
                    break
                s ^= 1 << bits[int(rng.integers(len(bits)))]
            ahead, behind = _closure(mask, N, [s], True), _closure(mask, N, [s], False)
            if not (ahead & ~behind).any():
                break
        found.append((np.flatnonzero(ahead), behind))
        left &= ~behind
    return found


def _blocks(states, mask, N, rates):
    """K restricted to `states`, one dense matrix per rate set: K[t, s] = rate of s -> t, out-rates on the diagonal."""
    pos = np.full(1 << N, -1, dtype=np.int64)
    pos[states] = np.arange(len(states))
    K = torch.zeros((len(rates), len(states), len(states)), dtype=torch.float64, device="cuda")
    r = torch.from_numpy(rates).cuda()
    for i in range(N):
        s = states[(mask[states] >> i & 1) == 1]
        t = pos[s ^ (1 << i)]
        code = torch.from_numpy(2 * i + (s >> i & 1)).cuda()
        p = torch.from_numpy(pos[s]).cuda()
        K[:, p, p] -= r[:, code]
        inside = torch.from_numpy(t >= 0).cuda()
        K[:, torch.from_numpy(t[t >= 0]).cuda(), p[inside]] = r[:, code[inside]]
    return K


def _stationary(net, rates):
    """[sets][2^N] limits of exp(K t) x0, or None where the dense systems would take too long."""
    N, n = net.N, 1 << net.N
    mask = _flip_masks(net)
    start = _start(net)
    x0 = np.where(start, 1.0 / start.sum(), 0.0)
    reach = _closure(mask, N, np.flatnonzero(start), True)
    parts = _terminal_components(mask, N, reach)
    count = np.sum([behind for _, behind in parts], axis=0)
    undecided = np.flatnonzero(reach & (count > 1))
    sizes = [len(states) for states, _ in parts] + [len(undecided)]
    if max(sizes) > 6000 or sum(0.7 * k ** 3 for k in sizes) * len(rates) > 2.5e12:
        return None
    out = torch.zeros((len(rates), n), dtype=torch.float64, device="cuda")
    chunk = max(1, min(len(rates), int(2e8) // max(max(sizes), 1) ** 2))
    for c in range(0, len(rates), chunk):
        r = rates[c:c + chunk]
        rd = torch.from_numpy(r).cuda()
        mass = [torch.full((len(r),), float(x0[behind & (count == 1)].sum()), dtype=torch.float64, device="cuda")
                for _, behind in parts]
        if len(undecided):
            # time spent in the undecided states: K_uu y = -x0; what leaves them goes to one component each
            b = torch.from_numpy(-x0[undecided]).cuda().expand(len(r), -1).unsqueeze(-1).contiguous()
            y = torch.linalg.solve(_blocks(undecided, mask, N, r), b).squeeze(-1)
            for i in range(N):
                go = (mask[undecided] >> i & 1) == 1
                src = undecided[go]
                flow = y[:, torch.from_numpy(np.flatnonzero(go)).cuda()] * rd[:, torch.from_numpy(2 * i + (src >> i & 1)).cuda()]
                dst = src ^ (1 << i)
                for k, (_, behind) in enumerate(parts):
                    to = np.flatnonzero(behind[dst] & (count[dst] == 1))
                    if to.size:
                        mass[k] += flow[:, torch.from_numpy(to).cuda()].sum(1)
        for (states, _), m in zip(parts, mass):
            pi = torch.ones((len(r), 1), dtype=torch.float64, device="cuda")
            if len(states) > 1:
                A = _blocks(states, mask, N, r)
                A[:, -1, :] = 1.0
                b = torch.zeros((len(r), len(states), 1), dtype=torch.float64, device="cuda")
                b[:, -1] = 1.0
                pi = torch.linalg.solve(A, b).squeeze(-1)
            out[c:c + chunk, torch.from_numpy(states).cuda()] = pi * m[:, None]
    return out


def _mlp_forward64(params, x):
    """Activations per layer and the softmax of the last, GELU in its tanh form."""
    acts, h = [], x.double()
    for l in range(0, len(params), 2):
        acts.append(h)
        z = h @ params[l] + params[l + 1]
        h = torch.nn.functional.gelu(z, approximate="tanh") if l + 2 < len(params) else z
    return torch.softmax(h, 1), h


def _train64(case, seed):
    params, x, t = _mlp_inputs(case, seed)
    params = [p.double().requires_grad_() for p in params]
    m = [torch.zeros_like(p) for p in params]
    v = [torch.zeros_like(p) for p in params]
    rows, steps, losses = case["rows"], case["steps"], []
    for j in range(steps):
        _, logits = _mlp_forward64(params, x[j * rows:(j + 1) * rows])
        loss = -(t[j * rows:(j + 1) * rows].double() * torch.log_softmax(logits, 1)).sum(1).mean()
        losses.append(loss.item())
        lr = LR_FIRST * (LR_LAST / LR_FIRST) ** (j / max(steps - 1, 1))
        with torch.no_grad():
            for k, g in enumerate(torch.autograd.grad(loss, params)):
                m[k] = 0.9 * m[k] + 0.1 * g
                v[k] = 0.999 * v[k] + 0.001 * g * g
                mh, vh = m[k] / (1 - 0.9 ** (j + 1)), v[k] / (1 - 0.999 ** (j + 1))
                params[k] -= lr * mh / (vh.sqrt() + 1e-8)
    return {"loss": float(np.mean(losses)),
            "params": torch.cat([p.detach().reshape(-1) for p in params]).cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        params, x, _ = _mlp_inputs(case, seed)
        return {"probs": _mlp_forward64([p.double() for p in params], x)[0]}
    if kind == "train":
        return _train64(case, seed)
    finals = [_stationary(net, r) for net, r in zip(_networks(case), _rates(case, seed))]
    if all(f is None for f in finals):
        return None
    if kind == "pipeline":
        return {"final": finals[0][0].cpu().numpy(), "order": None, "offsets": None, "scc": None, "terminals": None}
    return {"final": finals}
