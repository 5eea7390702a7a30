"""Performance cases: the calls a program makes into this package, over the sizes it is used at.

A case names a workload kind, an instance of the repository's banded family (``instances.Instance``: n qubits, band,
graph seed, optional phase gadgets), a storage type and how many strings one call takes.  Kinds:

  sample   exact samples of one in-place plan (``Engine.sample``)
  prob     log2 Pr of given strings, table renormalised every step (``Engine.prob``)
  chain    log2 Pr, conditionals and amplitude of given strings (``Engine.chain``)
  hybrid   a forced prefix (ancillas on 0, the first data bits given), the rest sampled (``Engine.hybrid``)
  score    many strings of one or several plans in one batch (``BatchEngine.score``)
  grad     gradients of every amplitude with respect to every measurement matrix (``BatchEngine.grad``)
  tt_sample, tt_chain   the two-table engine (``TwoTableEngine``)

``prepare`` holds what such a program keeps between calls (the engine with its plan) and the call's own inputs, made
from the seed.  ``exact`` evaluates the same linear-rank-width recurrence in 64 bits with plain torch on the plan's
gather records, one string (or lane) after the other.
"""
import functools
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests"))
from _pkg import egs  # noqa: E402

gs = egs.gsamp
_tmp = tempfile.TemporaryDirectory(prefix="gs_cases_")


def listed():
    return [
        # one shot of a small circuit: the smallest call there is, launches and latency
        dict(name="sample_n24_one", kind="sample", n=24, band=10, gseed=1, storage="c64", count=1),
        # probabilities of a file of strings of the same circuit in double storage (a check of a small device)
        dict(name="prob_n24_c128", kind="prob", n=24, band=10, gseed=1, storage="c128", count=64),
        # a batch of shots of a mid-size circuit
        dict(name="sample_n40", kind="sample", n=40, band=16, gseed=7, storage="c64", count=32),
        # proposals of the doped sampler: ancillas and a data prefix forced, the suffix sampled
        dict(name="hybrid_n48_doped", kind="hybrid", n=48, band=20, gseed=5, gadgets=12, forced=9, storage="c64", count=6),
        # scoring strings with conditionals, double storage
        dict(name="chain_n60_c128", kind="chain", n=60, band=24, gseed=4, storage="c128", count=12),
        # the benchmark's width-30 sampling configuration
        dict(name="sample_n70_b30", kind="sample", n=70, band=30, gseed=2, R=30, storage="c64", count=2),
        # scoring on a wide plan (width 29)
        dict(name="chain_n70_b32", kind="chain", n=70, band=32, gseed=3, storage="c64", count=2),
        # the largest arena of the list (width 31, 17 GB)
        dict(name="sample_n72_b35", kind="sample", n=72, band=35, gseed=3, storage="c64", count=1),
        # many small circuits scored together
        dict(name="score_mix", kind="score", n=33, band=13, gseed=2, storage="c64", lanes=128, plans=5),
        # batched scoring on the benchmark's band-26 instance
        dict(name="score_n70_b26", kind="score", n=70, band=26, gseed=3, storage="c64", lanes=64, plans=1),
        # a training step's forward and backward on the benchmark's gradient instance
        dict(name="grad_n60", kind="grad", n=60, band=24, gseed=4, storage="c64", lanes=128, plans=1),
        # the two-table sampler
        dict(name="tt_sample_n70_b30", kind="tt_sample", n=70, band=30, gseed=2, storage="c64", count=1),
    ]


# Most strings (or lanes) x 2^band of a drawn case, by kind: no drawn case costs more than the largest listed one.
_DRAW_LOG2 = dict(sample=31, prob=31, chain=31, hybrid=31, score=31, grad=30, tt_sample=30, tt_chain=30)


def draw(rng):
    kind = rng.choice(("sample", "sample", "prob", "chain", "hybrid", "score", "score", "grad", "tt_sample", "tt_chain"))
    most = _DRAW_LOG2[kind]
    storage = rng.choice(("c64", "c64", "c128"))
    case = dict(kind=kind, gseed=rng.randrange(1, 1000), storage=storage)
    if kind in ("score", "grad"):
        band = rng.randint(9, 25 if kind == "score" else 23)
        room = max(0, most - band - (storage == "c128") - 6)
        case.update(band=band, lanes=64 * (1 << rng.randint(0, min(room, 3))), plans=1)
        if kind == "score" and band <= 16:
            case["plans"] = rng.randint(1, 7)
    else:
        band = rng.randint(8, most - (storage == "c128"))
        count = 2 ** rng.uniform(0, min(6.0, most - band - (storage == "c128")))
        case.update(band=band, count=max(1, int(count)))
    case["n"] = rng.randint(band + 4, min(72, 3 * band + 8))
    if kind == "hybrid":
        case["gadgets"] = rng.choice((0, 0, rng.randint(1, 14)))
        case["forced"] = rng.randint(0, case["n"] // 2)
    return case


# ---- instances and plans (a program keeps them; one per circuit and process)

@functools.lru_cache(maxsize=64)
def _instance(n, band, gseed, gadgets, R):
    inst = egs.instances.Instance(n, band, gseed, R=R, gadgets_count=gadgets)
    path = os.path.join(_tmp.name, f"{n}_{band}_{gseed}_{gadgets}_{R}.txt")
    inst.write_plan(path)
    return inst, path


def _instances(case):
    return [_instance(case["n"] + 3 * i, case["band"] - (i % 3), case["gseed"] + i, case.get("gadgets", 0), case.get("R"))
            for i in range(case.get("plans", 1))]


def _tt_path(case, inst):
    path = os.path.join(_tmp.name, f"tt_{case['n']}_{case['band']}_{case['gseed']}.txt")
    if not os.path.exists(path):
        egs.engine.write_sampler_plan(path, inst.am)
    return path


def _strings(case, inst, seed, i=0):
    """The call's bit strings: uniform (a device's output looks uniform bit by bit); ancillas on 0."""
    rows = case["lanes"] if "lanes" in case else case["count"]
    b = np.random.default_rng([int(seed), i]).integers(0, 2, size=(rows, len(inst.steps))).astype(np.int8)
    anc = inst.N - inst.n
    b[:, :anc] = 0
    if case["kind"] == "hybrid":
        b[:, anc + case["forced"]:] = -1
    return b


def _call_seed(seed):
    return int(np.random.default_rng([int(seed), 77]).integers(1, 1 << 40))


def prepare(case, seed):
    kind = case["kind"]
    storage = gs.C64 if case["storage"] == "c64" else gs.C128
    insts = _instances(case)
    inst, path = insts[0]
    state = dict(case=case, seed=_call_seed(seed))
    if kind in ("score", "grad"):
        state["bits"] = [_strings(case, ins, seed, i) for i, (ins, _) in enumerate(insts)]
        state["engine"] = gs.BatchEngine([p for _, p in insts], [case["lanes"]] * len(insts), storage=storage)
    else:
        if kind not in ("sample", "tt_sample"):
            state["bits"] = _strings(case, inst, seed)
        state["engine"] = (gs.TwoTableEngine(_tt_path(case, inst), storage=storage) if kind.startswith("tt_")
                           else gs.Engine(path, storage))
    return state


def run(state):
    e, case = state["engine"], state["case"]
    kind = case["kind"]
    if kind in ("sample", "tt_sample"):
        bits, lp = e.sample(case["count"], state["seed"])
        return {"bits": bits, "log2p": lp}
    if kind == "prob":
        return {"log2p": e.prob(state["bits"])}
    if kind in ("chain", "tt_chain"):
        lp, cond, amp = e.chain(state["bits"])
        return {"log2p": lp, "cond": cond, "amp": amp}
    if kind == "hybrid":
        bits, lp, cond = e.hybrid(state["bits"], state["seed"])
        return {"bits": bits, "log2p": lp, "cond": cond}
    if kind == "score":
        lp, cond, amp = e.score(state["bits"])
        return {"log2p": lp, "cond": cond, "amp": amp}
    res, _ = e.grad(state["bits"])
    return {"log2p": [r[0] for r in res], "amp": [r[1] for r in res], "grad": [r[2] for r in res]}


def work(case):
    """One read of every step's table and one write of the next one, per string (a gradient: the same forward, then
    one read of every table and one read and write of the adjoint's); per written entry two complex products, their
    sum and |.|^2."""
    esz = 8 if case["storage"] == "c64" else 16
    rows = case["lanes"] if "lanes" in case else case["count"]
    entries_in = sum(2.0 ** s["r"] for inst, _ in _instances(case) for s in inst.am.steps)
    entries_out = sum(2.0 ** s["rn"] for inst, _ in _instances(case) for s in inst.am.steps)
    if case["kind"] == "grad":
        return {"bytes": rows * esz * (3 * entries_in + 2 * entries_out), "flops": rows * (18 * entries_out + 48 * entries_in)}
    return {"bytes": rows * esz * (entries_in + entries_out), "flops": rows * (18 * entries_out + 4 * entries_in)}


# ---- the same values in 64 bits

class _Mt64:
    """std::mt19937_64 and uniform_real_distribution<double>(0, 1) (one 64-bit word per draw, / 2^64)."""

    def __init__(self, seed):
        m = (1 << 64) - 1
        x = [seed & m]
        for i in range(1, 312):
            x.append((6364136223846793005 * (x[-1] ^ (x[-1] >> 62)) + i) & m)
        self.x, self.i = x, 312

    def uniform(self):
        x = self.x
        if self.i == 312:
            for i in range(312):
                y = (x[i] & 0xFFFFFFFF80000000) | (x[(i + 1) % 312] & 0x7FFFFFFF)
                x[i] = x[(i + 156) % 312] ^ (y >> 1) ^ (0xB5026F5AA96619E9 if y & 1 else 0)
            self.i = 0
        y = x[self.i]
        self.i += 1
        y ^= (y >> 29) & 0x5555555555555555
        y ^= (y << 17) & 0x71D67FFFEDA60000
        y ^= (y << 37) & 0xFFF7EEE000000000
        y &= (1 << 64) - 1
        return float(y ^ (y >> 43)) / 2.0 ** 64


def _spread(lo, hi, pos, device):
    """Addresses of the outputs lo .. hi - 1: bit j of the output goes to bit pos[j]."""
    cp = torch.arange(lo, hi, dtype=torch.int64, device=device)
    a = torch.zeros_like(cp)
    for j, p in enumerate(pos):
        a |= ((cp >> j) & 1) << p
    return a


def _span(ker):
    v = [0]
    for x in ker:
        v += [y ^ x for y in v]
    return v


def _odd(v):
    for s in (32, 16, 8, 4, 2, 1):
        v = v ^ (v >> s)
    return (v & 1).bool()


def _gathers(s, lo, hi, device):
    """(index, x, sign) of every input of the outputs lo .. hi - 1 of one plan record."""
    base = _spread(lo, hi, s["piv"], device)
    low = (1 << s["r"]) - 1
    for k in _span(s["ker"]):
        u = base ^ k
        c = u & low
        x = ((u >> s["r"]) & 1).bool()
        yield c, x, torch.where(_odd(c & s["rho"]) & x, -1.0, 1.0).to(torch.float64)


_CHUNK = 1 << 25


def _sums(s, old, lo, hi):
    """Signed sums of the x = 0 and of the x = 1 inputs of the outputs lo .. hi - 1; old: [entries, lanes]."""
    S = [torch.zeros((hi - lo, old.shape[1]), dtype=torch.complex128, device=old.device) for _ in range(2)]
    for c, x, sign in _gathers(s, lo, hi, old.device):
        v = old[c] * sign[:, None]
        S[0] += torch.where(x[:, None], 0, v)
        S[1] += torch.where(x[:, None], v, 0)
    return S


def _parts(s, lanes):
    n, step = 1 << s["rn"], max(1, _CHUNK // lanes)
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _norms(t):
    return torch.view_as_real(t).square().sum(dim=(0, 2))


def _walk_string(inst, bits, draws, device):
    """One string (a negative bit is sampled: U < p1): bits, log2 Pr, conditionals, the last entry."""
    t = torch.ones((1, 1), dtype=torch.complex128, device=device)
    prev, logp, amp, out, cond = 1.0, 0.0, 1.0, [], []
    for k, s in enumerate(inst.am.steps):
        M = inst.am.M[s["v"]]
        b = int(bits[k]) if bits is not None else -1
        if b < 0:
            n = [0.0, 0.0]
            for lo, hi in _parts(s, 1):
                S = _sums(s, t, lo, hi)
                for i in range(2):
                    n[i] += float(_norms(complex(M[i, 0]) * S[0] + complex(M[i, 1]) * S[1])[0])
                del S
            b = int(draws.uniform() < n[1] / (n[0] + n[1]))
        new = torch.empty((1 << s["rn"], 1), dtype=torch.complex128, device=device)
        for lo, hi in _parts(s, 1):
            S = _sums(s, t, lo, hi)
            new[lo:hi] = complex(M[b, 0]) * S[0] + complex(M[b, 1]) * S[1]
            del S
        nb = float(_norms(new)[0])
        out.append(b)
        cond.append(nb / (2 * prev))
        logp += math.log2(cond[-1]) if cond[-1] > 0 else -math.inf
        amp *= math.sqrt(nb)
        t = new.mul_(1 / math.sqrt(nb)) if nb > 0 else new
        prev = 1.0
    return out, logp, cond, complex(t[0, 0]) * amp


def _walk_lanes(inst, bits, device, grad):
    """All lanes of one plan at once: log2 Pr, conditionals, Z and (grad) dZ/dM_k[b_k, x]."""
    B = bits.shape[0]
    t = torch.ones((1, B), dtype=torch.complex128, device=device)
    prev = torch.ones(B, dtype=torch.float64, device=device)
    cond, kept, ws = [], [], []
    for k, s in enumerate(inst.am.steps):
        M = torch.from_numpy(np.asarray(inst.am.M[s["v"]], dtype=complex)).to(device)
        w = M[torch.from_numpy(bits[:, k].astype(np.int64)).to(device)]
        new = torch.empty((1 << s["rn"], B), dtype=torch.complex128, device=device)
        for lo, hi in _parts(s, B):
            S = _sums(s, t, lo, hi)
            new[lo:hi] = w[:, 0] * S[0] + w[:, 1] * S[1]
            del S
        if grad:
            kept.append(t)
            ws.append(w)
        nb = sum(_norms(new[lo:hi]) for lo, hi in _parts(s, B))
        cond.append(nb / (2 * prev))
        prev, t = nb, new
    lp = torch.log2(prev) - len(inst.am.steps)
    amp = t[0]
    if not grad:
        return lp, torch.stack(cond, 1), amp, None
    G = torch.empty((B, len(inst.am.steps), 2), dtype=torch.complex128, device=device)
    lam = torch.ones((1, B), dtype=torch.complex128, device=device)
    for k in reversed(range(len(inst.am.steps))):
        s, w, t = inst.am.steps[k], ws[k], kept.pop()
        back = torch.zeros_like(t)
        G[:, k] = 0
        for lo, hi in _parts(s, B):
            S = _sums(s, t, lo, hi)
            for x in range(2):
                G[:, k, x] += (lam[lo:hi] * S[x]).sum(0)
            del S
            for c, x, sign in _gathers(s, lo, hi, device):
                back.index_add_(0, c, lam[lo:hi] * sign[:, None] * torch.where(x[:, None], w[:, 1], w[:, 0]))
        lam = back
    return lp, torch.stack(cond, 1), amp, G


def exact(case, seed):
    kind = case["kind"]
    insts = _instances(case)
    rows = case["lanes"] if "lanes" in case else case["count"]
    entries = rows * sum(2.0 ** s["rn"] for inst, _ in insts for s in inst.am.steps)
    if entries > 2.0 ** (33 if kind == "grad" else 36) or sum(inst.width for inst, _ in insts[:1]) > 31:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind in ("score", "grad"):
        got = []
        for i, (inst, _) in enumerate(insts):
            bits = _strings(case, inst, seed, i)
            parts = [_walk_lanes(inst, bits[a:a + 16], device, kind == "grad") for a in range(0, rows, 16)]
            got.append([None if p[0] is None else torch.cat(p).cpu().numpy() for p in zip(*parts)])
        if kind == "score":
            return {"log2p": [g[0] for g in got], "cond": [g[1] for g in got], "amp": [g[2] for g in got]}
        return {"log2p": [g[0] for g in got], "amp": [g[2] for g in got], "grad": [g[3] for g in got]}
    inst = insts[0][0]
    bits = None if kind in ("sample", "tt_sample") else _strings(case, inst, seed)
    walks = [_walk_string(inst, None if bits is None else bits[i], _Mt64(_call_seed(seed) + i), device) for i in range(rows)]
    out = {"log2p": np.array([w[1] for w in walks])}
    if kind in ("sample", "tt_sample", "hybrid"):
        out["bits"] = np.array([w[0] for w in walks], dtype=np.int8)
    if kind in ("chain", "tt_chain", "hybrid"):
        out["cond"] = np.array([w[2] for w in walks])
    if kind in ("chain", "tt_chain"):
        out["amp"] = np.array([w[3] for w in walks])
    return out
