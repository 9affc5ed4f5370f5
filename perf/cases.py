"""Workloads of the alignment framework, for timing it and comparing its results.

A case is a dict of plain values.  Four families, by the public entry point
that serves them:

* ``solutions``: ``GlobalSolver`` / ``SemiglobalSolver`` / ``LocalSolver``
  ``.solve`` on problem objects over str sequences, ``Solution`` codomain:
  scores, paths and alignments.
* ``scores``: the core solver's ``solve_ragged`` on symbol codes that already
  sit in GPU memory, score only: database search and all-against-all.
* ``align_grad``: ``torch_ops.align_score`` forward and backward.
* ``dtw_grad``: ``torch_ops.dtw_distance`` forward and backward.
"""

import math

import numpy as np
import torch

import pyalign_amd as pa
from pyalign_amd import algorithm
from pyalign_amd.torch_ops import align_score, dtw_distance

LETTERS = "ACDEFGHIKLMNPQRSTVWY"
DNA = "ACGT"
SOLVERS = {"global": pa.GlobalSolver, "semiglobal": pa.SemiglobalSolver, "local": pa.LocalSolver}
LOCALITIES = {"global": algorithm.Locality.GLOBAL, "semiglobal": algorithm.Locality.SEMIGLOBAL,
              "local": algorithm.Locality.LOCAL}


def _seqs(name, family, n, s, t, spread="uniform", form="table", locality="local", gap="affine", g0=10.0, g1=1.0,
          direction="maximize"):
    c = {"family": family, "n": n, "lo_s": s[0], "hi_s": s[1], "lo_t": t[0], "hi_t": t[1], "spread": spread,
         "form": form, "locality": locality, "gap": gap, "g0": g0, "g1": g1, "direction": direction}
    return {"name": name, **c} if name else c


def listed():
    dna = dict(form="binary", locality="global", gap="linear", g0=0.2, g1=0.0)
    return [
        # an interactive call: one pair of words, the README's example
        _seqs("words_pair", "solutions", 1, (8, 8), (8, 8), **dna),
        # plain global alignment of a bag of short DNA strings, with paths
        _seqs("dna_bag", "solutions", 4096, (100, 100), (100, 100), **dna),
        # a read placed in a contig: one long semiglobal pair, with its path
        _seqs("long_pair", "solutions", 1, (5045, 5045), (10000, 10000), form="binary", locality="semiglobal",
              g0=2.0, g1=0.5),
        # the hits of a protein search aligned: local Gotoh with paths
        _seqs("protein_hits", "solutions", 2048, (50, 2000), (50, 2000), "log"),
        # general (logarithmic) gap costs: a bag of domains, and one pair
        _seqs("log_gap_bag", "solutions", 1024, (100, 300), (100, 300), gap="log", g0=3.0, g1=1.0),
        _seqs("log_gap_pair", "solutions", 1, (1200, 1200), (1000, 1000), locality="global", gap="log", g0=3.0, g1=1.0),
        # edit distances of many word pairs (minimise, unit costs)
        _seqs("edit_distances", "scores", 65536, (4, 24), (4, 24), form="binary", locality="global", gap="linear",
              g0=1.0, g1=0.0, direction="minimize"),
        # reads against reference windows: semiglobal affine scores
        _seqs("read_windows", "scores", 16384, (100, 150), (200, 400), form="binary", locality="semiglobal",
              g0=2.0, g1=0.5),
        # global affine scores of protein pairs (a distance matrix)
        _seqs("protein_global", "scores", 16384, (50, 1000), (50, 1000), "log", locality="global"),
        # protein search: local Gotoh scores of a whole bag
        _seqs("protein_search", "scores", 65536, (50, 2000), (50, 2000), "log"),
        # a training step through differentiable global affine alignment
        {"name": "align_train", "family": "align_grad", "n": 1024, "lo": 64, "hi": 512, "locality": "global",
         "gap": "affine", "g0": 1.0, "g1": 0.2},
        # a training step through DTW of long trajectories
        {"name": "dtw_train", "family": "dtw_grad", "n": 8192, "lo": 128, "hi": 4096, "dim": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above (odd sizes, other localities, gap
    models, forms and directions)."""
    family = rng.choice(["solutions", "solutions", "log_gap", "scores", "scores", "align_grad", "dtw_grad"])
    if family == "align_grad":
        hi = _log(rng, 24, 700)
        n = min(_log(rng, 4, 1024), int(2.6e8 / hi ** 2))
        gap = rng.choice(["affine", "linear"])
        return {"family": family, "n": n, "lo": max(2, hi // rng.randint(2, 8)), "hi": hi,
                "locality": rng.choice(["global", "semiglobal", "local"]), "gap": gap,
                "g0": rng.choice([0.5, 1.0, 1.5]), "g1": 0.2 if gap == "affine" else 0.0}
    if family == "dtw_grad":
        hi = _log(rng, 48, 4096)
        n = min(_log(rng, 8, 8192), int(8e10 / hi ** 2))
        return {"family": family, "n": n, "lo": max(2, hi // rng.randint(2, 32)), "hi": hi, "dim": rng.randint(1, 4)}
    if family == "log_gap":
        n = _log(rng, 1, 1024)
        most = (1.4e9 * min(n, 40) / n) ** (1 / 3)  # one pair uses less of the GPU than a bag
        hs, ht = (max(8, min(_log(rng, 30, 1200), int(most))) for _ in range(2))
        form = rng.choice(["table", "binary"])
        return _seqs(None, "solutions", n, (max(2, hs // 3), hs), (max(2, ht // 3), ht), form=form,
                     locality=rng.choice(["global", "semiglobal", "local"]), gap="log",
                     g0=rng.choice([1.5, 2.0, 3.0]), g1=rng.choice([0.5, 1.0]))
    single = family == "solutions" and rng.random() < 0.4
    most = {"solutions": 3e9, "scores": 1.6e10}[family]
    if single:
        n = 1
        hs, ht = _log(rng, 5, 7000), _log(rng, 5, 7000)
        ls, lt = hs, ht
    else:
        n = _log(rng, 16, 4096 if family == "solutions" else 65536)
        hs, ht = _log(rng, 12, 2000), _log(rng, 12, 2000)
        if n * hs * ht > 4 * most:
            n = int(4 * most / (hs * ht))
        ls, lt = max(2, hs // rng.randint(1, 40)), max(2, ht // rng.randint(1, 40))
    form = rng.choice(["table", "binary"])
    gap = rng.choice(["affine", "linear"])
    g0, g1 = rng.choice([(10.0, 1.0), (8.0, 2.0)] if form == "table" else [(2.0, 0.5), (3.0, 1.0)])
    if gap == "linear":
        g0, g1 = (4.0 if form == "table" else rng.choice([0.2, 1.0])), 0.0
    locality = rng.choice(["global", "semiglobal", "local"])
    direction = "minimize" if locality == "global" and form == "binary" and rng.random() < 0.4 else "maximize"
    return _seqs(None, family, n, (ls, hs), (lt, ht), rng.choice(["uniform", "log"]), form, locality, gap, g0, g1,
                 direction)


# ---- inputs ------------------------------------------------------------------

def _lengths(rng, n, lo, hi, spread):
    if spread == "log":
        x = np.floor(np.exp(rng.uniform(math.log(lo), math.log(hi), n)))
    else:
        x = rng.integers(lo, hi + 1, n)
    return np.clip(x, lo, hi).astype(np.int32)


def _table(rng):
    """Symmetric integer substitution scores of 20 symbols."""
    t = rng.integers(-4, 4, size=(20, 20))
    t = np.triu(t) + np.triu(t, 1).T
    np.fill_diagonal(t, rng.integers(4, 12, size=20))
    return t.astype(np.float32)


def _offsets(lens):
    off = np.zeros(len(lens), np.int64)
    off[1:] = np.cumsum(lens[:-1], dtype=np.int64)
    return off


def _sequences(case, seed):
    """Lengths, offsets and flat codes (on the GPU).  Every other pair is
    related: t follows s with substitutions and one insertion or deletion."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    ls = _lengths(rng, n, case["lo_s"], case["hi_s"], case["spread"])
    lt = _lengths(rng, n, case["lo_t"], case["hi_t"], case["spread"])
    table = _table(rng)
    if case["direction"] == "minimize":
        table = -table
    symbols = 4 if case["form"] == "binary" else 20
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    s = torch.randint(0, symbols, (int(ls.sum()),), generator=g, device=dev)
    t = torch.randint(0, symbols, (int(lt.sum()),), generator=g, device=dev)
    off_s, off_t = _offsets(ls), _offsets(lt)

    def per_symbol(x):
        return torch.repeat_interleave(torch.as_tensor(x, device=dev), torch.as_tensor(lt, device=dev).long())

    j = torch.arange(len(t), device=dev) - per_symbol(off_t)
    start = rng.integers(-10, 11, n) + np.where(ls > lt, rng.integers(0, 1 << 30, n) % np.maximum(ls - lt, 1),
                                               -(rng.integers(0, 1 << 30, n) % np.maximum(lt - ls, 1)))
    at = j + per_symbol(start) + torch.where(j > per_symbol(lt // 2), per_symbol(rng.integers(-6, 7, n)), 0)
    related = per_symbol((np.arange(n) % 2 == 0)) & (at >= 0) & (at < per_symbol(ls))
    related &= torch.rand(len(t), generator=g, device=dev) < (0.9 if case["form"] == "binary" else 0.6)
    src = s[(at + per_symbol(off_s)).clamp(0, len(s) - 1)]
    t = torch.where(related, src, t)
    return ls, lt, off_s, off_t, s, t, table


def _gap_cost(case):
    if case["gap"] == "log":
        return pa.LogarithmicGapCost(case["g0"], case["g1"])
    if case["gap"] == "affine":
        return pa.AffineGapCost(case["g0"], case["g1"])
    return pa.LinearGapCost(case["g0"])


def _binary_values(case):
    return (1, -1) if case["direction"] == "maximize" else (0, 1)


def _walks(case, seed):
    """Two batches of Gaussian random walks (steps N(0, 0.1^2)), padded."""
    rng = np.random.default_rng(seed)
    n, hi, dim = case["n"], case["hi"], case["dim"]
    lx, ly = (_lengths(rng, n, case["lo"], hi, "uniform") for _ in range(2))
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for lens in (lx, ly):
        w = (torch.randn(n, hi, dim, generator=g, device="cuda") * 0.1).cumsum(1)
        live = torch.arange(hi, device="cuda")[None, :] < torch.as_tensor(lens, device="cuda")[:, None]
        out.append(w * live[:, :, None])
    return lx, ly, out[0], out[1]


def _embeddings(case, seed):
    """Similarities of N(0, 1) / 8 embeddings of 64 dimensions, [n, hi, hi]."""
    rng = np.random.default_rng(seed)
    n, hi = case["n"], case["hi"]
    ls, lt = (_lengths(rng, n, case["lo"], hi, "uniform") for _ in range(2))
    g = torch.Generator(device="cuda").manual_seed(seed)
    a, b = (torch.randn(n, hi, 64, generator=g, device="cuda") / 8 for _ in range(2))
    return ls, lt, torch.bmm(a, b.transpose(1, 2).contiguous())


def prepare(case, seed):
    family = case["family"]
    if family == "solutions":
        ls, lt, off_s, off_t, s, t, table = _sequences(case, seed)
        letters = DNA if case["form"] == "binary" else LETTERS
        byte = np.frombuffer(letters.encode("latin-1"), dtype=np.uint8)
        text_s, text_t = (byte[x.cpu().numpy()].tobytes().decode("latin-1") for x in (s, t))
        if case["form"] == "binary":
            eq, ne = _binary_values(case)
            factory = pa.binary(eq=eq, ne=ne, direction=case["direction"])
        else:
            pairs = {(x, y): float(table[i, j]) for i, x in enumerate(letters) for j, y in enumerate(letters)}
            factory = pa.alphabetic(list(letters), lambda x, y: pairs[(x, y)], direction=case["direction"])
        problems = [factory.new_problem(text_s[a:a + m], text_t[b:b + k])
                    for a, m, b, k in zip(off_s.tolist(), ls.tolist(), off_t.tolist(), lt.tolist())]
        return {"family": family, "problems": problems if case["n"] > 1 else problems[0],
                "most": case["n"] * (case["hi_s"] + case["hi_t"] + 1),
                "solver": SOLVERS[case["locality"]](gap_cost=_gap_cost(case), codomain=pa.Solution)}
    if family == "scores":
        ls, lt, off_s, off_t, s, t, table = _sequences(case, seed)
        opts = algorithm.m16.create_options(dict(
            solver=algorithm.Type.ALIGNMENT, batch=True, return_dup=False, codomain=pa.solve.Codomain(pa.Score),
            direction=algorithm.Direction.__members__[case["direction"].upper()],
            locality=LOCALITIES[case["locality"]], gap_cost=_gap_cost(case)))
        binary = case["form"] == "binary"
        s, t = (x.to(torch.int32 if binary else torch.uint8) for x in (s, t))
        payload = dict(codes_s=s.data_ptr(), codes_t=t.data_ptr(), off_s=off_s, off_t=off_t, on_device=True)
        if binary:
            payload["eq"], payload["ne"] = _binary_values(case)
        else:
            payload["table"] = table
        return {"family": family, "solver": algorithm.m16.create_solver(case["hi_s"], case["hi_t"], opts),
                "form": "binary" if binary else "indexed", "ls": ls, "lt": lt, "payload": payload, "keep": (s, t)}
    if family == "align_grad":
        ls, lt, S = _embeddings(case, seed)
        return {"family": family, "S": S.requires_grad_(True), "ls": ls, "lt": lt, "locality": case["locality"],
                "gap": case["gap"], "open": torch.tensor(case["g0"], requires_grad=True),
                "extend": torch.tensor(case["g1"], requires_grad=True)}
    lx, ly, x, y = _walks(case, seed)
    return {"family": family, "x": x.requires_grad_(True), "y": y.requires_grad_(True), "lx": lx, "ly": ly}


# ---- one pass ------------------------------------------------------------------

def _laid_out(arrays, rows, *columns):
    """The arrays one after the other, at the start of an array of the case's largest size."""
    out = np.zeros((rows, *columns), dtype=np.int32)
    if arrays:
        np.concatenate(arrays, out=out[:sum(map(len, arrays))])
    return out


def run(state):
    family = state["family"]
    if family == "solutions":
        got = state["solver"].solve(state["problems"])
        if not isinstance(got, list):
            got = [got]
        found = [x for x in got if x.score is not None]  # (a local problem may have no alignment)
        paths = [x.path for x in found]
        return {"scores": np.array([x.score if x.score is not None else 0.0 for x in got], dtype=np.float32),
                "lengths": _laid_out([np.array([len(p) for p in paths])], len(got)),
                "paths": _laid_out(paths, state["most"], 2),
                "s_to_t": _laid_out([x.alignment.s_to_t for x in found], state["most"])}
    if family == "scores":
        return {"scores": state["solver"].solve_ragged("score", state["form"], state["ls"], state["lt"],
                                                       **state["payload"])}
    if family == "align_grad":
        S, go, ge = state["S"], state["open"], state["extend"]
        S.grad = go.grad = ge.grad = None
        scores = align_score(S, state["ls"], state["lt"], go, ge, locality=state["locality"], gap=state["gap"])
        scores.sum().backward()
        out = {"scores": scores.detach(), "dS": S.grad, "d_open": go.grad}
        if state["gap"] == "affine":
            out["d_extend"] = ge.grad
        return out
    x, y = state["x"], state["y"]
    x.grad = y.grad = None
    dist = dtw_distance(x, y, state["lx"], state["ly"])
    dist.sum().backward()
    return {"distances": dist.detach(), "dx": x.grad, "dy": y.grad}


# ---- what a pass cannot do without -----------------------------------------------

def _mean(lo, hi, spread="uniform"):
    return (hi - lo) / math.log(hi / lo) if spread == "log" and hi > lo else (lo + hi) / 2


def work(case):
    n = case["n"]
    if case["family"] == "dtw_grad":
        m = _mean(case["lo"], case["hi"])
        return {"bytes": n * (2 * m + 2 * case["hi"]) * case["dim"] * 4 + 4 * n,
                "flops": n * m * m * (3 * case["dim"] + 2)}
    if case["family"] == "align_grad":
        m = _mean(case["lo"], case["hi"])
        return {"bytes": n * (m * m + case["hi"] ** 2) * 4 + 4 * n,
                "flops": n * m * m * (9 if case["gap"] == "affine" else 6)}
    s = _mean(case["lo_s"], case["hi_s"], case["spread"])
    t = _mean(case["lo_t"], case["hi_t"], case["spread"])
    symbol = 4 if case["form"] == "binary" else 1
    out = 4 * n
    if case["family"] == "solutions":
        out += n * (max(s, t) * 8 + s * 4)  # path cells (two indices each) and s_to_t
    per_cell = {"linear": 6, "affine": 9, "log": s + t}[case["gap"]]  # log: an add and a max for every origin
    return {"bytes": n * (s + t) * symbol + out, "flops": n * s * t * per_cell}


# ---- the same results in 64 bits -------------------------------------------------

MOST_CELLS = 9e10  # padded cells of one exact() call (more would take too long)


def _flipped(t, Ls):
    """[n, Lt, ...] reversed and padded so that a diagonal's t values are one slice."""
    pad = t.new_zeros((t.shape[0], Ls) + t.shape[2:])
    return torch.cat([pad, t.flip(1), pad], 1)


class _Sweep:
    """The recurrences in float64 over one batch of problems, anti-diagonal by
    anti-diagonal (maximising; a minimising problem comes with its
    similarities negated)."""

    def __init__(self, ls, lt, gap, g0, g1, locality, keep):
        self.ls, self.lt = (torch.as_tensor(np.asarray(x), device="cuda").long() for x in (ls, lt))
        self.Ls, self.Lt = int(max(ls)), int(max(lt))
        self.gap, self.g0, self.g1, self.locality, self.keep = gap, g0, g1, locality, keep
        self.n = len(ls)

    def border(self, k):
        if k == 0:
            return 0.0
        if self.gap == "dtw":
            return -math.inf
        if self.locality != "global":
            return 0.0
        return -self.g0 * k if self.gap == "linear" else -(self.g0 + self.g1 * (k - 1))

    def run(self, similarity):
        """similarity(d): [n, Ls], values of the cells (i, d - i), i = 1 .. Ls."""
        n, Ls, Lt = self.n, self.Ls, self.Lt
        full = dict(dtype=torch.float64, device="cuda")
        D1 = torch.full((n, Ls + 1), -math.inf, **full)
        D2 = D1.clone()
        P, Q = D1.clone(), D1.clone()
        D2[:, 0] = self.border(0)
        D1[:, 0] = D1[:, 1] = self.border(1)
        best = torch.full((n,), -math.inf, **full)
        rows = torch.arange(1, Ls + 1, device="cuda")[None, :]
        self.codes = [None, None]
        for d in range(2, Ls + Lt + 1):
            dg = D2[:, :-1] + similarity(d)
            if self.gap == "affine":
                po, pe, qo, qe = D1[:, :-1] - self.g0, P[:, :-1] - self.g1, D1[:, 1:] - self.g0, Q[:, 1:] - self.g1
                up, left = torch.maximum(po, pe), torch.maximum(qo, qe)
            elif self.gap == "linear":
                up, left = D1[:, :-1] - self.g0, D1[:, 1:] - self.g0
            else:  # dtw: the cost is added after the choice
                dg, up, left, cost = D2[:, :-1], D1[:, :-1], D1[:, 1:], similarity(d)
            new = torch.maximum(torch.maximum(dg, up), left)
            if self.keep:
                code = torch.where(dg >= new, 1, torch.where(up >= new, 2, 3)).to(torch.int8)
                if self.gap == "affine":
                    code += (pe > po).to(torch.int8) * 4 + (qe > qo).to(torch.int8) * 8
                if self.locality == "local":
                    code = torch.where(new > 0, code, 0).to(torch.int8)
                self.codes.append(code)
            if self.gap == "dtw":
                new = new + cost
            if self.locality == "local":
                new = new.clamp(min=0.0)
            D2, D1, old = D1, torch.empty_like(D1), D1
            D1[:, 1:] = new
            D1[:, 0] = self.border(d)
            if d <= Ls:
                D1[:, d] = self.border(d)
            if self.gap == "affine":
                P, Q = torch.full_like(old, -math.inf), torch.full_like(old, -math.inf)
                P[:, 1:], Q[:, 1:] = up, left
                if d <= Ls:
                    P[:, d] = Q[:, d] = -math.inf
            if self.locality == "global":
                best = torch.where(self.ls + self.lt == d, D1.gather(1, self.ls[:, None])[:, 0], best)
                continue
            live = (rows <= self.ls[:, None]) & (d - rows <= self.lt[:, None]) & (rows < d)
            if self.locality == "semiglobal":
                live &= (rows == self.ls[:, None]) | (d - rows == self.lt[:, None])
            best = torch.maximum(best, torch.where(live, new, -math.inf).amax(1))
        return best

    def walk(self, emit):
        """Follows the kept codes of global problems; emit(k, i, j, moved) for
        every cell (1-based) that is matched.  Returns gap runs and extensions."""
        n = self.n
        k = torch.arange(n, device="cuda")
        i, j, state = self.ls.clone(), self.lt.clone(), torch.zeros_like(self.ls)
        runs, longer = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.zeros(n, dtype=torch.float64, device="cuda")
        codes = torch.stack(self.codes[2:])
        for _ in range(self.Ls + self.Lt):
            live = (i > 0) & (j > 0)
            if not bool(live.any()):
                break
            c = codes[(i + j - 2).clamp(min=0), k, (i - 1).clamp(min=0)].long()
            move = torch.where(state == 0, c & 3, state)
            opened = live & (state == 0) & (move > 1)
            emit(k, i, j, live & (torch.ones_like(live) if self.gap == "dtw" else move == 1))
            if self.gap == "affine":
                ext = live & (move > 1) & (((c >> move) & 1) == 1)
                longer += ext
                state = torch.where(ext, move, 0)
            runs += opened
            i, j = i - (live & (move != 3)).long(), j - (live & (move != 2)).long()
        rest = i + j
        if self.gap == "linear":
            runs += rest
        else:
            runs += rest > 0
            longer += (rest - 1).clamp(min=0)
        return runs, longer


def _buckets(ls, lt, most):
    """Problems of similar shape together, at most `most` padded cells each."""
    key = np.ceil(np.log2(np.maximum(ls, 1))) * 64 + np.ceil(np.log2(np.maximum(lt, 1)))
    for v in np.unique(key):
        at = np.nonzero(key == v)[0]
        step = max(1, int(most / (float(ls[at].max()) * (ls[at].max() + lt[at].max()))))
        for q in range(0, len(at), step):
            yield at[q:q + step]


def _padded(flat, off, lens, at):
    m = int(lens[at].max())
    ix = torch.as_tensor(off[at], device="cuda")[:, None] + torch.arange(m, device="cuda")[None, :]
    return flat[ix.clamp(max=len(flat) - 1)]


def _exact_scores(case, seed):
    ls, lt, off_s, off_t, s, t, table = _sequences(case, seed)
    sign = 1.0 if case["direction"] == "maximize" else -1.0
    out = np.zeros(case["n"])
    weights = torch.as_tensor(table, device="cuda").double() * sign
    eq, ne = (sign * x for x in _binary_values(case))
    if case["form"] == "binary":
        weights = torch.full((4, 4), ne, dtype=torch.float64, device="cuda")
        weights.fill_diagonal_(eq)
    flat, K = weights.flatten(), weights.shape[0]
    for at in _buckets(ls, lt, 4e9):
        a, b = _padded(s, off_s, ls, at), _padded(t, off_t, lt, at)
        if case["gap"] == "log":
            out[at] = _general(weights, a, b, ls[at], lt[at], case).cpu().numpy()
            continue
        sweep = _Sweep(ls[at], lt[at], case["gap"], case["g0"], case["g1"], case["locality"], False)
        a, b, Ls, Lt = a * K, _flipped(b, sweep.Ls), sweep.Ls, sweep.Lt
        best = sweep.run(lambda d: flat[a + b[:, Ls + Lt - d + 1:2 * Ls + Lt - d + 1]])
        out[at] = best.cpu().numpy()
    return torch.as_tensor(out * sign)


def _general(weights, a, b, ls, lt, case):
    """General gap costs: every origin of a gap, anti-diagonal by anti-diagonal."""
    n, Ls, Lt = len(ls), a.shape[1], b.shape[1]
    full = dict(dtype=torch.float64, device="cuda")
    k = np.arange(1, max(Ls, Lt) + 2)
    w = np.concatenate([[0.0], case["g0"] + case["g1"] * np.log(k)])
    edge = -w if case["locality"] == "global" else np.zeros_like(w)
    W = np.full((max(Ls, Lt) + 1,) * 2, -np.inf)  # W[x, y] = -w(x - y), y < x
    x, y = np.tril_indices(len(W), -1)
    W[x, y] = -w[x - y]
    W, edge = torch.as_tensor(W, **full), torch.as_tensor(edge, **full)
    D = torch.full((n, Ls + 1, Lt + 1), -math.inf, **full)  # by row, and transposed
    D[:, :, 0], D[:, 0, :] = edge[:Ls + 1], edge[:Lt + 1]
    T = D.transpose(1, 2).contiguous()
    for d in range(2, Ls + Lt + 1):
        i = torch.arange(max(1, d - Lt), min(Ls, d - 1) + 1, device="cuda")
        j = d - i
        new = D[:, i - 1, j - 1] + weights[a[:, i - 1], b[:, j - 1]]
        new = torch.maximum(new, (T[:, j, :] + W[i, :Ls + 1]).amax(2))
        new = torch.maximum(new, (D[:, i, :] + W[j, :Lt + 1]).amax(2))
        if case["locality"] == "local":
            new = new.clamp(min=0.0)
        D[:, i, j] = T[:, j, i] = new
    ls, lt = (torch.as_tensor(v, device="cuda").long() for v in (ls, lt))
    if case["locality"] == "global":
        return D[torch.arange(n, device="cuda"), ls, lt]
    i, j = torch.arange(Ls + 1, device="cuda")[None, :, None], torch.arange(Lt + 1, device="cuda")[None, None, :]
    li, lj = ls[:, None, None], lt[:, None, None]
    live = (i >= 1) & (j >= 1) & (i <= li) & (j <= lj)
    if case["locality"] == "semiglobal":
        live &= (i == li) | (j == lj)
    return torch.where(live, D, -math.inf).amax((1, 2))


def _exact_align(case, seed):
    ls, lt, S = _embeddings(case, seed)
    S = S.double()
    n, hi, path = case["n"], case["hi"], case["locality"] == "global"
    scores = torch.zeros(n, dtype=torch.float64)
    dS = torch.zeros(S.shape, dtype=torch.float64, device="cuda") if path else None
    d_open = d_ext = 0.0
    for at in _buckets(ls, lt, 2e9):
        sweep = _Sweep(ls[at], lt[at], case["gap"], case["g0"], case["g1"], case["locality"], path)
        Ls, Lt, m = sweep.Ls, sweep.Lt, len(at)
        part = S[torch.as_tensor(at, device="cuda"), :Ls, :Lt].contiguous()

        def similarity(d):
            lo, hi_ = max(1, d - Lt), min(Ls, d - 1)
            out = part.new_zeros((m, Ls))
            cells = part.as_strided((m, hi_ - lo + 1), (Ls * Lt, Lt - 1), (lo - 1) * Lt + d - lo - 1)
            out[:, lo - 1:hi_] = cells
            return out

        scores[torch.as_tensor(at)] = sweep.run(similarity).cpu()
        if path:
            ix = torch.as_tensor(at, device="cuda")

            def emit(k, i, j, on):
                dS.view(-1).index_add_(0, (ix[k] * hi * hi + (i - 1).clamp(min=0) * hi + (j - 1).clamp(min=0)),
                                       on.double())

            runs, longer = sweep.walk(emit)
            d_open, d_ext = d_open - float(runs.sum()), d_ext - float(longer.sum())
    out = {"scores": scores, "dS": dS, "d_open": np.float64(d_open) if path else None}
    if case["gap"] == "affine":
        out["d_extend"] = np.float64(d_ext) if path else None
    return out


def _exact_dtw(case, seed):
    lx, ly, x, y = _walks(case, seed)
    x, y = x.double(), y.double()
    dist = torch.zeros(case["n"], dtype=torch.float64)
    dx, dy = torch.zeros_like(x), torch.zeros_like(y)
    for at in _buckets(lx, ly, 1e10):
        sweep = _Sweep(lx[at], ly[at], "dtw", 0.0, 0.0, "global", True)
        Ls, Lt, dim = sweep.Ls, sweep.Lt, case["dim"]
        ix = torch.as_tensor(at, device="cuda")
        a, b = x[ix, :Ls], y[ix, :Lt]
        f = _flipped(b, Ls)
        dist[torch.as_tensor(at)] = -sweep.run(
            lambda d: -(a - f[:, Ls + Lt - d + 1:2 * Ls + Lt - d + 1]).square().sum(2)).cpu()
        gx, gy = torch.zeros_like(a), torch.zeros_like(b)

        def emit(k, i, j, on):
            i, j = (i - 1).clamp(min=0), (j - 1).clamp(min=0)
            g = 2 * (a[k, i] - b[k, j]) * on[:, None]
            gx.view(-1, dim).index_add_(0, k * Ls + i, g)
            gy.view(-1, dim).index_add_(0, k * Lt + j, -g)

        sweep.walk(emit)
        dx[ix, :Ls], dy[ix, :Lt] = gx, gy
    return {"distances": dist, "dx": dx, "dy": dy}


def exact(case, seed):
    if case["family"] == "dtw_grad":
        return _exact_dtw(case, seed) if case["n"] * case["hi"] ** 2 < 2 * MOST_CELLS else None
    if case["family"] == "align_grad":
        return _exact_align(case, seed)
    if case["n"] * float(case["hi_s"]) * case["hi_t"] > MOST_CELLS * (40 if case["spread"] == "log" else 1):
        return None
    scores = _exact_scores(case, seed)
    if case["family"] == "scores":
        return {"scores": scores}
    return {"scores": scores, "lengths": None, "paths": None, "s_to_t": None}
