"""Performance cases of the engine: the calls that a direct-optimization
tree search makes, through the package's public entry points.

Every case is a dict of plain values with a "kind":

  call    one pair of host sequences, synchronous (engine.Align): what POY's
          unchanged OCaml does through the stubs
  level   one tree level: a few pairs of medians in host memory, aligned in
          one call (engine.run_pair_list), as treepass does per level
  pairs   a batch of pairs resident on the device (engine.PairPlan): the
          joins and medians of a TBR round, and the batch workloads
  triples a batch of three-way alignments on the device (engine.TriplePlan)
  fitch   down and up pass over a tree's nonadditive characters, one call per
          tree level (poyg_fitch_down_w / poyg_fitch_up_w)
  powell  Powell's three-way search on one triple (engine.powell_3d), the
          readjustment of an Iterative ThreeD pass
  score   the model stage of a guided TBR round: 4-mer profiles of the
          medians, pair features, the network's predictions
  train   training of the join scorer: one pass over its rows with Adam
"""
import math

import numpy as np
import torch

from poyd_amd import engine, seqstore, surrogate, synth

GAP = 16
MODES = {"linear-cost": engine.POYG_MODE_LINEAR_COST, "linear-align": engine.POYG_MODE_LINEAR_ALIGN,
         "affine-cost": engine.POYG_MODE_AFFINE_COST, "affine-align": engine.POYG_MODE_AFFINE_ALIGN}
_context = None


def context():
    """The program's one device context."""
    global _context
    if _context is None:
        _context = engine.Context(0)
    return _context


def listed():
    return [
        # the smallest call: one join distance of a 300 bp locus from the OCaml side
        dict(name="call-cost-300", kind="call", op="cost", model="linear", length=300, sub=0.10),
        # one affine alignment with its medians of a 1 kb gene, per call
        dict(name="call-affine-1000", kind="call", op="align", model="affine", length=1000, sub=0.10),
        # a level of the 128-taxon build: a few pairs of ambiguous medians of 300-1,500 bp
        dict(name="level-linear-6", kind="level", model="linear", n=6, lmin=300, lmax=1500, sub=0.10),
        # the batch workload of short loci: 1,000 pairs of 200-400 bp, aligned with medians
        dict(name="linear-align-1000", kind="pairs", mode="linear-align", n=1000, lmin=200, lmax=400, sub=0.10),
        # join distances of a TBR round: loci of 500-2,000 bp, costs only
        dict(name="joins-linear-16384", kind="pairs", mode="linear-cost", n=16384, lmin=500, lmax=2000, sub=0.10),
        # the headline batch: 65,536 affine alignments of 50-5,000 bp with medians
        dict(name="affine-align-65536", kind="pairs", mode="affine-align", n=65536, lmin=50, lmax=5000, sub=0.18),
        # three-way alignments of the median batch, 100-500 bp
        dict(name="triples-1024", kind="triples", n=1024, lmin=100, lmax=500, sub=0.15),
        # a genome-scale matrix of nonadditive characters over 1,024 taxa
        dict(name="fitch-1024x1Mi", kind="fitch", taxa=1024, chars=1 << 20, width=1),
        # an ordinary morphology-and-sites matrix: 128 taxa, ten thousand characters, a number no power of two divides
        dict(name="fitch-128x10001", kind="fitch", taxa=128, chars=10001, width=1),
        # one readjustment of an Iterative ThreeD pass, 300 bp
        dict(name="powell-300", kind="powell", length=300, sub=0.10),
        # the model stage of a guided TBR round: a million candidate pairs
        dict(name="score-1Mi", kind="score", seqs=3000, n=1 << 20),
        # training the join scorer
        dict(name="train-131072", kind="train", n=131072, batch=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "call", "level", "pairs", "pairs", "pairs", "triples", "fitch", "fitch", "powell",
                       "score", "train"])
    sub = round(rng.uniform(0.05, 0.25), 3)
    if kind == "call":
        op, model = rng.choice([("cost", "linear"), ("align", "linear"), ("cost", "affine"), ("align", "affine")])
        return dict(kind=kind, op=op, model=model, length=_log(rng, 60, 2000), sub=sub)
    if kind == "level":
        lmin = _log(rng, 100, 600)
        return dict(kind=kind, model=rng.choice(["linear", "linear", "affine"]), n=_log(rng, 2, 64), lmin=lmin,
                    lmax=_log(rng, lmin + 50, 2000), sub=sub)
    if kind == "pairs":
        lmin = _log(rng, 50, 700)
        lmax = _log(rng, lmin + 50, 4000)
        # no more cells than the largest listed batches
        most = min(65536, int(3e9 / (lmax * (200 + 0.15 * lmax))))
        return dict(kind=kind, mode=rng.choice(sorted(MODES)), n=_log(rng, 64, max(most, 128)), lmin=lmin, lmax=lmax,
                    sub=sub)
    if kind == "triples":
        lmin = _log(rng, 40, 200)
        return dict(kind=kind, n=_log(rng, 8, 1000), lmin=lmin, lmax=_log(rng, lmin + 30, 450), sub=sub)
    if kind == "fitch":
        width = rng.choice([1, 1, 2, 4])
        taxa = _log(rng, 16, 1024)
        most = min(1 << 20, (1 << 28) // (taxa * width))
        return dict(kind=kind, taxa=taxa, chars=_log(rng, 500, most), width=width)
    if kind == "powell":
        return dict(kind=kind, length=_log(rng, 60, 320), sub=round(rng.uniform(0.04, 0.12), 3))
    if kind == "score":
        return dict(kind=kind, seqs=_log(rng, 200, 3000), n=_log(rng, 2000, 1 << 20))
    return dict(kind=kind, n=_log(rng, 8192, 131072), batch=rng.choice([1000, 2048, 4096, 4096]))


# ---------------------------------------------------------------- inputs
class Seqs:
    """Concatenated sequences with their leading gaps: `seq` on the GPU,
    offsets, lengths and gap counts on the host."""

    def __init__(self, body, ln, gen, amb=0.0, gap=0.0):
        n = len(ln)
        total = ln + 1
        off = torch.zeros(n, dtype=torch.int64, device="cuda")
        off[1:] = torch.cumsum(total, 0)[:-1]
        seq = torch.full((int(total.sum()),), GAP, dtype=torch.uint8, device="cuda")
        owner = torch.repeat_interleave(torch.arange(n, device="cuda"), ln)
        x = torch.bitwise_left_shift(torch.ones_like(body), body).to(torch.uint8)
        if amb or gap:   # medians: some positions hold a second base or the gap beside the base
            second = torch.randint(0, 4, (len(x),), generator=gen, device="cuda", dtype=torch.uint8)
            second = torch.bitwise_left_shift(torch.ones_like(second), second)
            x = torch.where(torch.rand(len(x), generator=gen, device="cuda") < amb, x | second, x)
            x = torch.where(torch.rand(len(x), generator=gen, device="cuda") < gap, x | GAP, x)
        seq[torch.arange(len(x), device="cuda") + owner + 1] = x
        gaps = torch.ones(n, dtype=torch.int64, device="cuda")
        gaps.index_add_(0, owner, ((x & GAP) != 0).to(torch.int64))
        self.seq, self.off, self.ln = seq, off.cpu().numpy(), total.to(torch.int32).cpu().numpy()
        self.gaps = gaps.to(torch.int32).cpu().numpy()

    def host(self):
        flat = self.seq.cpu().numpy()
        return [flat[o:o + m].copy() for o, m in zip(self.off.tolist(), self.ln.tolist())]


def _lengths(case, gen, n):
    """n lengths of the case's range, spread over their logarithm where it is
    wide: the same ones for every seed, in an order of its own."""
    lo, hi = case["lmin"], case["lmax"]
    u = (torch.randperm(n, generator=gen, device="cuda").double() + 0.5) / n
    if hi > 10 * lo:
        return torch.round(torch.exp(math.log(lo) + u * math.log(hi / lo))).to(torch.int64)
    return lo + torch.floor(u * (hi - lo + 1)).to(torch.int64)


def _room(plan, case, members):
    """Device bytes for the plan's outputs: enough for every seed's descendants."""
    lo, hi = case["lmin"], case["lmax"]
    need = plan.slots * case["n"] * int(members * 1.1 * _mean_power(lo, hi, 1) + 96)
    return torch.zeros(max(need, 1 << 20), dtype=torch.uint8, device="cuda")


def _roots(ln, gen):
    return torch.randint(0, 4, (int(ln.sum()),), generator=gen, device="cuda", dtype=torch.uint8)


def _mutate(root, ln, sub, gen):
    """Descendants: substitutions at rate `sub` per site, indel starts at a
    fifth of it, geometric lengths, half of them insertions."""
    n, total = len(ln), len(root)
    owner = torch.repeat_interleave(torch.arange(n, device="cuda"), ln)
    end = torch.cumsum(ln, 0)[owner]

    def rand():
        return torch.rand(total, generator=gen, device="cuda")

    out = torch.where(rand() < sub, (root + torch.randint(1, 4, (total,), generator=gen, device="cuda",
                                                          dtype=torch.uint8)) & 3, root)
    start = rand() < sub / 5
    is_ins = rand() < 0.5
    size = 1 + torch.floor(torch.log2(1 / rand().clamp_min(1e-6))).to(torch.int64)
    pos = torch.nonzero(start & ~is_ins).reshape(-1)
    diff = torch.zeros(total + 1, dtype=torch.int64, device="cuda")
    diff.index_add_(0, pos, torch.ones_like(pos))
    stop = torch.minimum(pos + size[pos], end[pos])
    diff.index_add_(0, stop, -torch.ones_like(stop))
    keep = torch.cumsum(diff[:-1], 0) == 0
    count = torch.where(start & is_ins, size, torch.zeros_like(size)) + keep
    site = torch.repeat_interleave(torch.arange(total, device="cuda"), count)
    last = (torch.cumsum(count, 0) - 1)[site] == torch.arange(len(site), device="cuda")
    ins = torch.randint(0, 4, (len(site),), generator=gen, device="cuda", dtype=torch.uint8)
    body = torch.where(last & keep[site], out[site], ins)
    return body, torch.zeros(n, dtype=torch.int64, device="cuda").index_add_(0, owner, count)


def _matrix(model):
    return (engine.CostMatrix.of_sub_indel(1, 2) if model == "linear" else engine.CostMatrix.of_sub_indel(1, 1, 3))


def _pair_seqs(case, seed, n, amb=0.0, gap=0.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ln = (torch.full((n,), case["length"], dtype=torch.int64, device="cuda") if "length" in case
          else _lengths(case, gen, n))
    root = _roots(ln, gen)
    a = Seqs(root, ln, gen, amb, gap)
    return a, Seqs(*_mutate(root, ln, case["sub"], gen), gen, amb, gap)


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# ------------------------------------------------------- call, level, pairs
def _prepare_call(case, seed):
    a, b = _pair_seqs(case, seed, 1)
    return dict(align=engine.Align(context()), cm=_matrix(case["model"]), a=a.host()[0], b=b.host()[0])


def _fixed(x, size):
    """x at the front of `size` zeros, and its length: outputs of one size whatever the inputs."""
    out = np.zeros(size, np.uint8)
    out[:len(x)] = x
    return out, len(x)


def _run_call(s):
    if s["case"]["op"] == "cost":
        return s["align"].cost_2(s["a"], s["b"], s["cm"])
    size = 3 * s["case"]["length"] + 64
    if s["case"]["model"] == "affine":
        med, ri, rj, cost, mwg = s["align"].align_affine_3(s["a"], s["b"], s["cm"])
        return [cost] + [_fixed(x, size) for x in (med, ri, rj, mwg)]
    ra, rb, cost = s["align"].align_2(s["a"], s["b"], s["cm"])
    return [cost] + [_fixed(x, size) for x in (ra, rb)]


def _prepare_level(case, seed):
    a, b = _pair_seqs(case, seed, case["n"], amb=0.04, gap=0.03)
    return dict(cm=_matrix(case["model"]), pairs=list(zip(a.host(), b.host())))


def _run_level(s):
    r = engine.run_pair_list(context(), s["cm"], MODES[s["case"]["model"] + "-align"], s["pairs"])
    size = s["case"]["n"] * (3 * s["case"]["lmax"] + 64)
    return [r.cost, r.out_len] + [_fixed(np.concatenate(r.seqs(k)), size) for k in range(r.slots)]


def _prepare_pairs(case, seed):
    a, b = _pair_seqs(case, seed, case["n"])
    model, op = case["mode"].split("-")
    cm = _matrix(model)
    seq = torch.cat([a.seq, b.seq])
    dw = None
    if model == "linear":   # DOS.median's band, and DOS.distance's for the joins
        dif = np.maximum(8, np.abs(a.ln.astype(np.int64) - b.ln))
        dw = seqstore.band_deltaw(a.ln, b.ln, a.gaps, b.gaps, dif if op == "cost" else None)
    plan = engine.PairPlan(context(), cm, MODES[case["mode"]], a.off, a.ln, b.off + len(a.seq), b.ln, dw)
    s = dict(plan=plan, seq=seq, cost=torch.zeros(case["n"], dtype=torch.int32, device="cuda"))
    if plan.slots:
        s["out"] = _room(plan, case, 2)
        assert s["out"].numel() >= plan.out_bytes
        s["out_len"] = torch.zeros(plan.slots * case["n"], dtype=torch.int32, device="cuda")
    return s


def _run_pairs(s):
    if "out" not in s:
        s["plan"].run(s["seq"].data_ptr(), s["cost"].data_ptr())
        return s["cost"]
    s["plan"].run(s["seq"].data_ptr(), s["cost"].data_ptr(), s["out"].data_ptr(), s["out_len"].data_ptr())
    return s["cost"], s["out"], s["out_len"]


# ----------------------------------------------------------------- triples
def _prepare_triples(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ln = _lengths(case, gen, case["n"])
    root = _roots(ln, gen)
    parts = [Seqs(*_mutate(root, ln, case["sub"], gen), gen) for _ in range(3)]
    seq = torch.cat([p.seq for p in parts])
    base = np.cumsum([0] + [len(p.seq) for p in parts])
    plan = engine.TriplePlan(context(), engine.CostMatrix3(_matrix("linear")),
                             *[x for q, p in enumerate(parts) for x in (p.off + base[q], p.ln)])
    out = _room(plan, case, 3)
    assert out.numel() >= plan.out_bytes
    return dict(plan=plan, seq=seq, cost=torch.zeros(case["n"], dtype=torch.int32, device="cuda"), out=out,
                out_len=torch.zeros(plan.slots * case["n"], dtype=torch.int32, device="cuda"))


# ------------------------------------------------------------------- fitch
def _prepare_fitch(case, seed):
    taxa, chars, width = case["taxa"], case["chars"], case["width"]
    rng = np.random.Generator(np.random.PCG64(seed))
    parent, _, leaves = synth.yule_tree(rng, taxa, 0.05)
    nodes = len(parent)
    kids = [[] for _ in range(nodes)]
    for v in range(1, nodes):
        kids[parent[v]].append(v)
    height, depth = np.zeros(nodes, np.int64), np.zeros(nodes, np.int64)
    for v in range(nodes - 1, 0, -1):
        height[parent[v]] = max(height[parent[v]], height[v] + 1)
    for v in range(1, nodes):
        depth[v] = depth[parent[v]] + 1
    inner = [v for v in range(nodes) if kids[v]]
    # rows: the preliminary sets of every node, then the final sets of the inner nodes (the root's are its preliminary ones)
    final = {v: nodes + q for q, v in enumerate(inner[1:])}
    final[0] = 0
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[width]
    states = torch.randint(2, 9 if width == 1 else 15, (chars,), generator=gen, device="cuda")
    rows = torch.zeros((nodes + len(inner) - 1, chars), dtype=kind, device="cuda")
    at = torch.from_numpy(leaves.astype(np.int64)).cuda()
    base = torch.randint(0, 1 << 20, (chars,), generator=gen, device="cuda")
    for k in range(0, len(leaves), 64):   # the taxa share half of their states
        m = at[k:k + 64]
        own = torch.randint(0, 1 << 20, (len(m), chars), generator=gen, device="cuda")
        same = torch.rand((len(m), chars), generator=gen, device="cuda") < 0.5
        rows[m] = torch.bitwise_left_shift(torch.ones_like(own), torch.where(same, base, own) % states).to(kind)
    down = [np.array([[kids[v][0], kids[v][1], v] for v in inner if height[v] == h], np.int32)
            for h in range(1, int(height.max()) + 1)]
    up = [np.array([[final[parent[v]], v, kids[v][0], kids[v][1], final[v]] for v in inner if depth[v] == d], np.int32)
          for d in range(1, int(depth.max()) + 1) if any(depth[v] == d for v in inner)]
    levels = []
    n_added = 0
    for jobs in down:
        levels.append((engine.load().poyg_fitch_down_w, len(jobs), _device(jobs.T), n_added))
        n_added += len(jobs)
    for jobs in up:
        levels.append((engine.load().poyg_fitch_up_w, len(jobs), _device(jobs.T), None))
    return dict(rows=rows, levels=levels, added=torch.zeros(n_added, dtype=torch.int64, device="cuda"))


def _run_fitch(s):
    ctx, width, chars = context(), s["case"]["width"], s["case"]["chars"]
    rows, added = s["rows"].data_ptr(), s["added"].data_ptr()
    engine.dev_zero(ctx, added, 8 * s["added"].numel())
    for call, n, jobs, at in s["levels"]:
        p = jobs.data_ptr()
        cols = [p + 4 * n * c for c in range(len(jobs))]
        if at is not None:
            cols.append(added + 8 * at)
        engine._check(call(ctx.h, width, rows, chars, n, *cols, None), "fitch level")
    return s["rows"], s["added"]


# ------------------------------------------------------------------ powell
def _prepare_powell(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ln = torch.tensor([case["length"]], device="cuda")
    root = _roots(ln, gen)
    return dict(seqs=[Seqs(*_mutate(root, ln, case["sub"], gen), gen).host()[0] for _ in range(3)])


def _run_powell(s):
    cost, aligned = engine.powell_3d(context(), *s["seqs"], 1, 2, 1)
    return [cost] + [_fixed(x, 5 * s["case"]["length"] + 64) for x in aligned]


# ------------------------------------------------------------ score, train
def _weights(seed):
    """He-uniform weights W1, b1, W2, b2, w3, b3 with small biases."""
    rng = np.random.Generator(np.random.PCG64(seed))
    bound = math.sqrt(6 / 256)
    sizes = [(256 * 256, bound), (256, 0.02), (256 * 256, bound), (256, 0.02), (256, bound), (1, 0.02)]
    return np.concatenate([rng.uniform(-b, b, k) for k, b in sizes]).astype(np.float32)


def _family(seed, n):
    """n related sequences of 500-2,000 bp (medians of one tree), on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ln = torch.randint(500, 2001, ((n + 7) // 8,), generator=gen, device="cuda")[torch.arange(n, device="cuda") // 8]
    group = torch.arange(n, device="cuda") // 8
    # eight descendants of each root: the root's bases repeated per descendant
    first = torch.cumsum(ln, 0) - ln
    owner = torch.repeat_interleave(torch.arange(n, device="cuda"), ln)
    site = torch.arange(int(ln.sum()), device="cuda") - first[owner]
    table = torch.randint(0, 4, (int(group.max()) + 1, 2001), generator=gen, device="cuda", dtype=torch.uint8)
    return Seqs(*_mutate(table[group[owner], site], ln, 0.1, gen), gen, 0.03, 0.02)


def _pair_index(seed, seqs, n):
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.integers(0, seqs, (2, n)).astype(np.int32)


def _prepare_score(case, seed):
    f = _family(seed, case["seqs"])
    sc = surrogate.Scorer(context(), 4096, 1)
    sc.set_params(_weights(seed))
    return dict(scorer=sc, seq=f.seq, off=_device(f.off), ln=_device(f.ln),
                counts=torch.zeros((case["seqs"], 256), device="cuda"),
                idx=_device(_pair_index(seed, case["seqs"], case["n"])),
                x=torch.zeros((case["n"], 256), dtype=torch.bfloat16, device="cuda"),
                y=torch.zeros(case["n"], device="cuda"))


def _run_score(s):
    lib, ctx, n = engine.load(), context(), s["case"]["n"]
    engine._check(lib.poyg_kmer_counts(ctx.h, s["seq"].data_ptr(), s["off"].data_ptr(), s["ln"].data_ptr(),
                                       s["case"]["seqs"], s["counts"].data_ptr(), None), "poyg_kmer_counts")
    p = s["idx"].data_ptr()
    engine._check(lib.poyg_pair_features(ctx.h, s["counts"].data_ptr(), p, p + 4 * n, n, surrogate.X_SCALE,
                                         s["x"].data_ptr(), None), "poyg_pair_features")
    s["scorer"].forward(s["x"].data_ptr(), n, s["y"].data_ptr())
    return s["counts"], s["x"], s["y"]


def _rows(case, seed):
    """Training rows: bf16 profile differences and targets that follow them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lam = 4 * torch.rand((1, 256), generator=gen, device="cuda")
    far = torch.rand((case["n"], 1), generator=gen, device="cuda")
    dif = torch.floor(lam * far * torch.randn((case["n"], 256), generator=gen, device="cuda").abs() * 3)
    t = far[:, 0] * 3 + 0.2 * torch.randn(case["n"], generator=gen, device="cuda")
    return (dif / 8).to(torch.bfloat16), t


def _order(n):
    """The permutation of Scorer.train's first epoch with seed 3."""
    return np.random.default_rng(3).permutation(n).astype(np.int32)


def _prepare_train(case, seed):
    x, t = _rows(case, seed)
    ctx = context()
    torch.cuda.synchronize()
    return dict(scorer=surrogate.Scorer(ctx, case["batch"], 1), weights=_weights(seed),
                x=engine.DeviceBuffer.from_array(ctx, x.view(torch.int16).cpu().numpy()),
                t=engine.DeviceBuffer.from_array(ctx, t.cpu().numpy()))


def _run_train(s):
    sc = s["scorer"]
    sc.set_params(s["weights"])
    losses = sc.train(s["x"], s["t"], s["case"]["n"], epochs=1, lr=1e-3, seed=3)
    return sc.params(), losses


_PREPARE = {"call": _prepare_call, "level": _prepare_level, "pairs": _prepare_pairs, "triples": _prepare_triples,
            "fitch": _prepare_fitch, "powell": _prepare_powell, "score": _prepare_score, "train": _prepare_train}
_RUN = {"call": _run_call, "level": _run_level, "pairs": _run_pairs, "triples": _run_pairs, "fitch": _run_fitch,
        "powell": _run_powell, "score": _run_score,
        "train": _run_train}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["case"] = case
    return s


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------- what a pass needs
def _mean_power(lo, hi, k):
    """Mean of L**k over the lengths of a case."""
    if hi > 10 * lo:
        return (hi ** k - lo ** k) / (k * math.log(hi / lo))
    return (hi ** (k + 1) - lo ** (k + 1)) / ((k + 1) * (hi - lo))


def _pair_work(model, align, n, l1, l2):
    """Pairs of mean length l1, mean squared length l2: 30 operations per
    cell of the affine band (about 85 columns), 8 per cell of the linear one
    (100 columns and 10% of the length)."""
    cells = n * 85 * l1 if model == "affine" else n * min(l2, 100 * l1 + 0.1 * l2)
    out = (4 if model == "affine" else 3) * n * 1.05 * l1 if align else 0
    return dict(bytes=2 * n * l1 + 4 * n + out, flops=cells * (30 if model == "affine" else 8))


def work(case):
    k = case["kind"]
    if k == "call":
        return _pair_work(case["model"], case["op"] == "align", 1, case["length"], case["length"] ** 2)
    if k in ("level", "pairs", "triples"):
        l1, l2, l3 = (_mean_power(case["lmin"], case["lmax"], p) for p in (1, 2, 3))
        n = case["n"]
        if k == "triples":
            return dict(bytes=n * (3 * l1 + 4 * 1.2 * l1 + 4), flops=20 * n * l3)
        model, align = (case["model"], True) if k == "level" else (case["mode"].split("-")[0],
                                                                  case["mode"].endswith("align"))
        return _pair_work(model, align, n, l1, l2)
    if k == "fitch":   # 3 rows per node of the down pass, 5 per node of the up pass; a dozen bit operations a byte
        b = case["chars"] * case["width"] * (3 * (case["taxa"] - 1) + 5 * (case["taxa"] - 2))
        return dict(bytes=b, flops=2 * b)
    if k == "powell":   # the search's cells grow with the cube of its cost, about half of the length
        return dict(bytes=6 * case["length"], flops=16 * 10 * (3 * case["sub"] * case["length"]) ** 3)
    if k == "score":
        n, m = case["n"], case["seqs"]
        return dict(bytes=1250 * m + 1024 * m + n * (8 + 512 + 4), flops=n * 2 * (2 * 256 * 256 + 256))
    n = case["n"] // case["batch"] * case["batch"]
    return dict(bytes=n * 516 + 4 * 132097 * 8, flops=n * 6 * (2 * 256 * 256 + 256))


def tolerance(case):
    """Alignments, costs and character sets are whole numbers.  The network's
    outputs: four times what the same roundings (bf16 operands and
    activations) with sums in another order gave (predictions 3.3e-5 and
    0.007, parameters after a training pass 7.4e-4 and 0.06)."""
    if case["kind"] == "score":
        return dict(rel=1.3e-4, max=0.03)
    if case["kind"] == "train":
        return dict(rel=3e-3, max=0.25)
    return "exact"


# ----------------------------------------------------------- 64-bit results
def _split(p):
    p = torch.from_numpy(p).cuda().double()
    cut = np.cumsum([0, 256 * 256, 256, 256 * 256, 256, 256, 1])
    w = [p[a:b].clone() for a, b in zip(cut[:-1], cut[1:])]
    w[0], w[2] = w[0].reshape(256, 256), w[2].reshape(256, 256)
    return w


def _net(x, w):
    h = torch.relu(torch.relu(x @ w[0] + w[1]) @ w[2] + w[3])
    return h @ w[4] + w[5]


def _exact_score(case, seed):
    f = _family(seed, case["seqs"])
    first = torch.from_numpy(f.off).cuda()
    owner = torch.repeat_interleave(torch.arange(case["seqs"], device="cuda"), torch.from_numpy(f.ln).cuda().long())
    base = torch.full((32,), -1, dtype=torch.int64)
    for v in range(32):   # the lowest base bit
        if v & 15:
            base[v] = (v & 15 & -(v & 15)).bit_length() - 1
    b = base.cuda()[f.seq.long()]
    win = torch.stack([b[k:len(b) - 3 + k] for k in range(4)])
    same = owner[:-3] == owner[3:]
    inside = torch.arange(len(b) - 3, device="cuda") > first[owner[:-3]]
    ok = same & inside & (win.min(0).values >= 0)
    code = owner[:-3] * 256 + win[0] * 64 + win[1] * 16 + win[2] * 4 + win[3]
    counts = torch.bincount(code[ok], minlength=256 * case["seqs"]).reshape(-1, 256).double()
    idx = torch.from_numpy(_pair_index(seed, case["seqs"], case["n"])).cuda().long()
    w = _split(_weights(seed))
    x = (counts[idx[0]] - counts[idx[1]]).abs() * surrogate.X_SCALE
    y = torch.cat([_net(x[r:r + 65536], w) for r in range(0, case["n"], 65536)])
    return counts, x, y


def _exact_train(case, seed):
    x, t = _rows(case, seed)
    order = torch.from_numpy(_order(case["n"])).cuda().long()
    w = [v.requires_grad_() for v in _split(_weights(seed))]
    m, v = [torch.zeros_like(p) for p in w], [torch.zeros_like(p) for p in w]
    losses, step = [], 0
    for r in range(0, case["n"] - case["batch"] + 1, case["batch"]):
        rows = order[r:r + case["batch"]]
        loss = torch.mean((_net(x[rows].double(), w) - t[rows].double()) ** 2)
        if step % 64 == 0:
            losses.append(float(loss.detach()))
        step += 1
        grads = torch.autograd.grad(loss, w)
        with torch.no_grad():
            for k, g in enumerate(grads):
                m[k] = 0.9 * m[k] + 0.1 * g
                v[k] = 0.999 * v[k] + 0.001 * g * g
                w[k] -= 1e-3 * (m[k] / (1 - 0.9 ** step)) / ((v[k] / (1 - 0.999 ** step)).sqrt() + 1e-8)
    params = torch.cat([p.detach().reshape(-1) for p in w])
    return params.cpu().numpy(), [sum(losses) / max(len(losses), 1)]


def exact(case, seed):
    if case["kind"] == "score":
        return _exact_score(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None
