"""GPU parity: every engine path against the CPU oracle, bit for bit.

All calls go through the C ABI (libpoyg.so).  Inputs are seeded; each case
prints its name before running so that a failing run names it.
"""
import sys

import numpy as np
import pytest

from poyd_amd import synth

pytestmark = pytest.mark.gpu
GAP = 16


@pytest.fixture(scope="module")
def ctx():
    from poyd_amd import engine
    try:
        return engine.Context(0)
    except engine.PoygError as e:
        pytest.skip(f"no GPU: {e}")


def note(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def batch_of(seqs):
    ln = np.array([len(s) for s in seqs], np.int32)
    off = np.zeros(len(seqs), np.int64)
    if len(seqs) > 1:
        off[1:] = np.cumsum(ln[:-1])
    return synth.SeqBatch(np.concatenate(seqs).astype(np.uint8) if seqs else np.zeros(0, np.uint8), off, ln)


def rand_seq(rng, n, alphabet="dna"):
    if alphabet == "dna":
        body = rng.choice([1, 2, 4, 8], size=n)
    elif alphabet == "ambig":
        body = rng.integers(1, 16, size=n)
    else:   # any 5-bit mask, gap-bearing symbols included
        body = rng.integers(1, 32, size=n)
    return np.concatenate([[GAP], body]).astype(np.uint8)


def mutate(rng, s, ps, pi):
    out = [GAP]
    for x in s[1:]:
        r = rng.random()
        if r < pi / 2:
            continue
        if r < pi:
            out.append(int(rng.choice([1, 2, 4, 8])))
        out.append(int(rng.choice([1, 2, 4, 8])) if rng.random() < ps else int(x))
    return np.array(out, np.uint8)


def mixed_pairs(rng, n, alphabet="dna"):
    A, B = [], []
    edge = [(0, 0), (0, 5), (7, 0), (1, 1), (39, 40), (40, 40), (41, 41), (45, 120), (300, 12), (10, 700),
            (700, 10), (250, 250), (1, 300)]
    for la, lb in edge:
        A.append(rand_seq(rng, la, alphabet))
        B.append(rand_seq(rng, lb, alphabet))
    for k in range(n):
        L = int(rng.integers(20, 600))
        a = rand_seq(rng, L, alphabet)
        b = mutate(rng, a, 0.2, 0.08) if k % 4 else rand_seq(rng, int(rng.integers(1, 600)), alphabet)
        if alphabet != "dna" and k % 2:
            b = rand_seq(rng, len(b) - 1, alphabet)
        A.append(a)
        B.append(b)
    return A, B


AFFINE_MATRICES = [(1, 1, 3), (2, 1, 1), (3, 1, 5)]


def test_concurrent_copies_agree(ctx, oracle):
    """Thousands of copies of a few wide-band pairs in one batch: every copy
    must give the oracle's result (many waves resident per workgroup)."""
    from poyd_amd import engine
    note("concurrent copies")
    rng = np.random.default_rng(31)
    base = [(rand_seq(rng, 388), rand_seq(rng, 542)), (rand_seq(rng, 300), rand_seq(rng, 420))]
    a0 = rand_seq(rng, 900)
    base.append((a0, mutate(rng, a0, 0.2, 0.06)))
    A = [base[k % 3][0] for k in range(3000)]
    B = [base[k % 3][1] for k in range(3000)]
    cm = engine.CostMatrix.of_sub_indel(1, 1, 3)
    ref = oracle.CM2.sub_indel(1, 1, 3)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    want = [oracle.align_affine_3(a, b, ref) for a, b in base]
    bad = [k for k in range(3000) if res.cost[k] != want[k % 3][3]]
    assert not bad, (len(bad), bad[:10])
    for k in range(0, 3000, 7):
        med, ri, rj, cost, mwg = want[k % 3]
        for slot, w in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), w), (k, slot)
    lcm = engine.CostMatrix.of_sub_indel(1, 2)
    lref = oracle.CM2.sub_indel(1, 2)
    res = engine.run_pairs(ctx, lcm, engine.POYG_MODE_LINEAR_ALIGN, batch_of(A), batch_of(B))
    lw = [oracle.align_2(a, b, lref) for a, b in base]
    bad = [k for k in range(3000) if res.cost[k] != lw[k % 3][0]]
    assert not bad, (len(bad), bad[:10])


@pytest.mark.parametrize("sub,indel,go", AFFINE_MATRICES)
@pytest.mark.parametrize("alphabet", ["dna", "any"])
def test_affine_batch_matches_oracle(ctx, oracle, sub, indel, go, alphabet):
    from poyd_amd import engine
    note(f"affine batch sub={sub} indel={indel} go={go} alphabet={alphabet}")
    rng = np.random.default_rng(100 + sub * 10 + go)
    A, B = mixed_pairs(rng, 120, alphabet)
    cm = engine.CostMatrix.of_sub_indel(sub, indel, go)
    ref = oracle.CM2.sub_indel(sub, indel, go)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    cres = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_COST, batch_of(A), batch_of(B))
    for k, (a, b) in enumerate(zip(A, B)):
        med, ri, rj, cost, mwg = oracle.align_affine_3(a, b, ref)
        assert res.cost[k] == cost, (k, len(a), len(b))
        assert cres.cost[k] == oracle.cost_affine_3(a, b, ref), (k, len(a), len(b))
        for slot, want in enumerate((med, mwg, ri, rj)):
            got = res.seq(k, slot)
            assert np.array_equal(got, want), (k, slot, len(a), len(b))


def block_indel_pairs(rng):
    """Pairs whose alignment path crosses many band lanes: long sequences
    with block insertions and deletions (band widths of 40 to 250 diagonal
    pairs), long runs of one state, several 1,024-step output batches, and
    sequences where one side ends early (tail gaps)."""
    A, B = [], []
    for k, (L, ins, dele) in enumerate([(1500, 150, 0), (1500, 0, 140), (2200, 300, 0), (900, 60, 60),
                                         (3000, 420, 30), (1200, 5, 5), (2500, 0, 0), (400, 200, 0),
                                         (1800, 90, 90), (700, 0, 380)]):
        a = rand_seq(rng, L)
        body = list(a[1:])
        if dele:
            at = int(rng.integers(0, L - dele))
            del body[at:at + dele]
        if ins:
            at = int(rng.integers(0, len(body)))
            body[at:at] = list(rng.choice([1, 2, 4, 8], size=ins))
        b = mutate(rng, np.array([GAP] + body, np.uint8), 0.1, 0.02)
        A.append(a)
        B.append(b)
        A.append(b)   # the same pair with the sides swapped
        B.append(a)
    return A, B


@pytest.mark.parametrize("sub,indel,go", AFFINE_MATRICES)
def test_affine_block_indels(ctx, oracle, sub, indel, go):
    from poyd_amd import engine
    note(f"affine block indels sub={sub} indel={indel} go={go}")
    rng = np.random.default_rng(700 + sub * 10 + go)
    A, B = block_indel_pairs(rng)
    cm = engine.CostMatrix.of_sub_indel(sub, indel, go)
    ref = oracle.CM2.sub_indel(sub, indel, go)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    for k, (a, b) in enumerate(zip(A, B)):
        med, ri, rj, cost, mwg = oracle.align_affine_3(a, b, ref)
        assert res.cost[k] == cost, (k, len(a), len(b))
        for slot, want in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), want), (k, slot, len(a), len(b))


@pytest.mark.parametrize("sub,indel,go", [(1, 1, 3), (2, 3, 1), (63, 2, 4), (64, 2, 4), (0, 1, 2)])
@pytest.mark.parametrize("alphabet", ["dna", "ambig"])
def test_affine_three_cost_groups(ctx, oracle, sub, indel, go, alphabet):
    """The steady groups of sequences without gap-bearing characters: lengths
    at which the first of them appear and end, bands at the last and first
    widths of 3 diagonal pairs a lane and of 1, 2 and 4 lane sets, one pair
    with a gap-bearing character among them, costs at and past the largest
    the form takes, in batches and per call."""
    from poyd_amd import engine
    note(f"affine three-cost groups sub={sub} indel={indel} go={go} alphabet={alphabet}")
    rng = np.random.default_rng(900 + sub + 7 * indel + 13 * go)
    pairs = []
    for n in (3, 4, 5, 20, 21, 22, 24, 29, 31, 38, 41, 42, 60, 99, 100, 101, 102, 103, 250):
        a = rand_seq(rng, n, alphabet)
        pairs.append((a, mutate(rng, a, 0.15, 0.06)))
    for diff in (46, 47, 48, 79, 80, 207, 208, 463):       # E0 = diff + 8
        a = rand_seq(rng, 420, alphabet)
        b = np.concatenate([a[:200], rand_seq(rng, diff, alphabet)[1:], a[200:]])
        pairs.append((a, mutate(rng, b, 0.1, 0.0)))
    gapped = pairs[18][0].copy()
    gapped[77] |= GAP
    A = [p[0] for p in pairs] * 2 + [gapped]
    B = [p[1] for p in pairs] * 2 + [pairs[18][1]]
    cm, ref = engine.CostMatrix.of_sub_indel(sub, indel, go), oracle.CM2.sub_indel(sub, indel, go)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    cost = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_COST, batch_of(A), batch_of(B)).cost
    al = engine.Align(ctx)
    for k, (a, b) in enumerate(zip(A, B)):
        med, ri, rj, want, mwg = oracle.align_affine_3(a, b, ref)
        assert res.cost[k] == want and cost[k] == oracle.cost_affine_3(a, b, ref), k
        for slot, w in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), w), (k, slot)
        if k < len(pairs):
            got = al.align_affine_3(a, b, cm)
            assert got[3] == want and all(np.array_equal(x, y) for x, y in zip(got[:3] + got[4:], (med, ri, rj, mwg))), k


def test_affine_wide_pairs_large_batch(ctx, oracle):
    """More pairs of two lane sets than three waves a SIMD hold (the fill's
    denser form), with and without gap-bearing characters."""
    from poyd_amd import engine
    note("affine wide pairs, large batch")
    rng = np.random.default_rng(940)
    A, B = [], []
    for k in range(40):
        a = rand_seq(rng, 100, "any" if k % 2 else "dna")
        A.append(a)
        B.append(np.concatenate([mutate(rng, a, 0.1, 0.0), rand_seq(rng, 72 + k)[1:]]))
    pick = np.concatenate([np.arange(40), rng.integers(0, 40, 3400)])
    cm, ref = engine.CostMatrix.of_sub_indel(1, 1, 3), oracle.CM2.sub_indel(1, 1, 3)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of([A[k] for k in pick]),
                           batch_of([B[k] for k in pick]))
    want = [oracle.align_affine_3(a, b, ref) for a, b in zip(A, B)]
    assert np.array_equal(res.cost, [want[k][3] for k in pick])
    for q, k in enumerate(pick):
        med, ri, rj, _, mwg = want[k]
        for slot, w in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(q, slot), w), (q, k, slot)


@pytest.mark.parametrize("sub,indel,go", [(1, 1, 1200000), (0, 1, 1000100), (1, 2500, 3), (63, 20000, 1),
                                          (1, 1, 333000), (1, 1400, 3)])
def test_affine_costs_past_closed_states(ctx, oracle, sub, indel, go):
    """Alignments that cost as much as the states the reference closes at the
    band's edges (HIGH_NUM, src/algn.c:38), and pairs on the other side of the
    rule for the three-cost groups: one, two and four lane sets, per call and in
    a batch; costs, and the alignment where the oracle's walk stays in the band."""
    from poyd_amd import engine
    note(f"affine costs past the closed states sub={sub} indel={indel} go={go}")
    rng = np.random.default_rng(910 + sub)
    A, B = [], []
    for la, lb in [(30, 30), (60, 75), (80, 110), (60, 160), (61, 300), (60, 505), (200, 290)]:
        if 2 * (la + lb + 4) * max(indel, go) + 3000000 >= 1 << 29:   # (refused by the plan)
            continue
        a = rand_seq(rng, la)
        A.append(a)
        B.append(np.concatenate([mutate(rng, a, 0.2, 0.0), rand_seq(rng, lb - la)[1:]]))
    cm, ref = engine.CostMatrix.of_sub_indel(sub, indel, go), oracle.CM2.sub_indel(sub, indel, go)
    want = [oracle.cost_affine_3(a, b, ref) for a, b in zip(A, B)]
    cost = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_COST, batch_of(A), batch_of(B)).cost
    assert list(cost) == want
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B), check_band=False)
    al = engine.Align(ctx)
    aligned = 0
    for k, (a, b) in enumerate(zip(A, B)):
        assert al.cost_2(a, b, cm) == want[k], k
        try:
            med, ri, rj, c, mwg = oracle.align_affine_3(a, b, ref)
        except RuntimeError:   # the reference reads outside its band
            continue
        aligned += 1
        assert res.cost[k] == c, k
        for slot, w in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), w), (k, slot)
        got = al.align_affine_3(a, b, cm)
        assert got[3] == c and all(np.array_equal(x, y) for x, y in zip(got[:3] + got[4:], (med, ri, rj, mwg))), k
    assert aligned


def test_affine_exact_band_width(ctx, oracle):
    """A batch whose direction bands pass 32 GiB keeps the exact band width (41
    diagonal pairs, not 42: the last lane stores its dwords one by one); every
    copy of the pair gives the oracle's alignment."""
    from poyd_amd import engine
    note("affine exact band width")
    rng = np.random.default_rng(71)
    a = rand_seq(rng, 5000)
    b = mutate(rng, a, 0.1, 0.0)
    n = (32 << 30) // (2501 * 4 * 42) + 1000
    cm, ref = engine.CostMatrix.of_sub_indel(1, 1, 3), oracle.CM2.sub_indel(1, 1, 3)
    ln = np.full(n, len(a), np.int32)
    plan = engine.PairPlan(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, np.zeros(n, np.int64), ln,
                           np.full(n, len(a), np.int64), ln)
    seq = engine.DeviceBuffer.from_array(ctx, np.concatenate([a, b]))
    cost, out, length = (engine.DeviceBuffer(ctx, size) for size in (4 * n, plan.out_bytes, 16 * n))
    plan.run(seq.ptr, cost.ptr, out.ptr, length.ptr)
    assert plan.status() == 0
    ctx.sync()
    med, ri, rj, want, mwg = oracle.align_affine_3(a, b, ref)
    assert (cost.download(np.int32, n) == want).all()
    lens, rows = length.download(np.int32, 4 * n).reshape(n, 4), out.download(np.uint8, plan.out_bytes).reshape(n, -1)
    cap = int(plan.cap[0])
    for slot, w in enumerate((med, mwg, ri, rj)):
        assert (lens[:, slot] == len(w)).all(), slot
        bad = (rows[:, (slot + 1) * cap - len(w):(slot + 1) * cap] != w).any(axis=1)
        assert not bad.any(), (slot, np.flatnonzero(bad)[:10])
    for buf in (seq, cost, out, length):
        buf.free()


@pytest.mark.parametrize("alphabet", ["dna", "any"])
def test_affine_packed_fill_saturation(ctx, oracle, alphabet):
    """The packed 16-bit narrow-band fill holds values as 4 v saturated at
    0xffff: pairs whose cost reaches 0x3fff are queued for the 32-bit fill.
    Costs of 40 / 30 / 50 put short DNA pairs below that bound and longer
    ones above it, in one batch; every output equals the oracle's and the
    32-bit fill's."""
    from poyd_amd import engine
    note(f"affine packed fill saturation alphabet={alphabet}")
    rng = np.random.default_rng(911 + (alphabet == "any"))
    A, B = [], []
    for k in range(96):
        L = int(rng.integers(20, 900))
        a = rand_seq(rng, L, alphabet)
        b = mutate(rng, a, 0.3, 0.05) if k % 3 else rand_seq(rng, L + int(rng.integers(-15, 15)), alphabet)
        A.append(a)
        B.append(b)
    cm = engine.CostMatrix.of_sub_indel(40, 30, 50)
    ref = oracle.CM2.sub_indel(40, 30, 50)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    cres = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_COST, batch_of(A), batch_of(B))
    ctx.set_tuning("aff_narrow_kernel", 1)
    try:
        res32 = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, batch_of(A), batch_of(B))
    finally:
        ctx.set_tuning("aff_narrow_kernel", -1)
    costs = []
    for k, (a, b) in enumerate(zip(A, B)):
        med, ri, rj, cost, mwg = oracle.align_affine_3(a, b, ref)
        costs.append(cost)
        assert res.cost[k] == cost and res32.cost[k] == cost, (k, len(a), len(b))
        assert cres.cost[k] == oracle.cost_affine_3(a, b, ref), (k, len(a), len(b))
        for slot, want in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), want), (k, slot, len(a), len(b))
            assert np.array_equal(res32.seq(k, slot), want), (k, slot, len(a), len(b))
    costs = np.array(costs)
    if alphabet == "dna":   # gap-bearing characters make the other alphabet's alignments cheap
        assert (costs < 0x3fff).sum() >= 10 and (costs >= 0x3fff).sum() >= 5, costs


@pytest.mark.parametrize("sub,indel", [(1, 2), (1, 1), (2, 1)])
@pytest.mark.parametrize("alphabet", ["dna", "ambig"])
def test_linear_batch_matches_oracle(ctx, oracle, sub, indel, alphabet):
    from poyd_amd import engine
    note(f"linear batch sub={sub} indel={indel} alphabet={alphabet}")
    rng = np.random.default_rng(200 + sub * 10 + indel)
    A, B = mixed_pairs(rng, 120, alphabet)
    cm = engine.CostMatrix.of_sub_indel(sub, indel)
    ref = oracle.CM2.sub_indel(sub, indel)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_ALIGN, batch_of(A), batch_of(B))
    cres = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_COST, batch_of(A), batch_of(B))
    for k, (a, b) in enumerate(zip(A, B)):
        cost, oa, ob = oracle.align_2(a, b, ref)
        assert res.cost[k] == cost, (k, len(a), len(b))
        assert cres.cost[k] == oracle.cost_2(a, b, ref), (k, len(a), len(b))
        assert np.array_equal(res.seq(k, 0), oa), (k, len(a), len(b))
        assert np.array_equal(res.seq(k, 1), ob), (k, len(a), len(b))
        assert np.array_equal(res.seq(k, 2), oracle.median_2(oa, ob, ref)), k


def test_linear_explicit_deltaw(ctx, oracle):
    """DOS.distance passes ?deltaw (src/seqCS.ml:856-866); the batch takes the
    resulting band parameter per pair."""
    from poyd_amd import engine
    note("linear explicit deltaw")
    rng = np.random.default_rng(7)
    A, B = mixed_pairs(rng, 40)
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    ref = oracle.CM2.sub_indel(1, 2)
    dws = [max(8, abs(len(a) - len(b))) for a, b in zip(A, B)]
    bands = np.array([engine.deltaw(a, b, d) for a, b, d in zip(A, B, dws)], np.int32)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_COST, batch_of(A), batch_of(B), bands)
    for k, (a, b) in enumerate(zip(A, B)):
        assert res.cost[k] == oracle.cost_2(a, b, ref, dws[k])


def test_linear_long_columns(ctx, oracle):
    """Column sequences around 2,048: the systolic kernel takes up to 2,048
    columns (a full-plane band of that width included), the row kernels
    longer ones (narrow bands in LDS rings, a wide full-plane band)."""
    from poyd_amd import engine
    note("linear long columns")
    rng = np.random.default_rng(11)
    shapes = [(2047, 2047), (2048, 2048), (2049, 2049), (2100, 2200), (3072, 2048), (3100, 2049), (3600, 2300)]
    A, B = [], []
    for la, lb in shapes:
        a = rand_seq(rng, la)
        b = mutate(rng, a, 0.15, 0.05)[:lb] if lb <= la else rand_seq(rng, lb)
        A.append(a)
        B.append(b)
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    ref = oracle.CM2.sub_indel(1, 2)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_ALIGN, batch_of(A), batch_of(B))
    cres = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_COST, batch_of(A), batch_of(B))
    for k, (a, b) in enumerate(zip(A, B)):
        cost, oa, ob = oracle.align_2(a, b, ref)
        assert res.cost[k] == cost, (k, len(a), len(b))
        assert cres.cost[k] == cost, (k, len(a), len(b))
        assert np.array_equal(res.seq(k, 0), oa), (k, len(a), len(b))
        assert np.array_equal(res.seq(k, 1), ob), (k, len(a), len(b))


def test_per_call_entry_points(ctx, oracle):
    from poyd_amd import engine
    note("per-call entry points")
    rng = np.random.default_rng(9)
    al = engine.Align(ctx)
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    ref = oracle.CM2.sub_indel(1, 2)
    cma = engine.CostMatrix.of_sub_indel(1, 1, 3)
    refa = oracle.CM2.sub_indel(1, 1, 3)
    # short pairs, then the lengths of the per-call benchmark and longer
    sizes = [int(rng.integers(1, 200)) for _ in range(12)] + [300, 300, 1000, 1000, 2500]
    for k, n in enumerate(sizes):
        a = rand_seq(rng, n)
        b = mutate(rng, a, 0.1, 0.05) if k % 2 else rand_seq(rng, n if n >= 300 else int(rng.integers(1, 200)))
        assert al.cost_2(a, b, cm) == oracle.cost_2(a, b, ref)
        x, y, c = al.align_2(a, b, cm)
        c2, ox, oy = oracle.align_2(a, b, ref)
        assert c == c2 and np.array_equal(x, ox) and np.array_equal(y, oy)
        got = al.align_affine_3(a, b, cma)
        want = oracle.align_affine_3(a, b, refa)
        assert got[3] == want[3]
        for g, w in zip(got, want):
            if isinstance(g, np.ndarray):
                assert np.array_equal(g, w)
        assert al.cost_2(a, b, cma) == oracle.cost_affine_3(a, b, refa)


def test_three_d_matches_oracle(ctx, oracle):
    import ctypes as C
    from poyd_amd import engine
    note("three-dimensional alignment")
    rng = np.random.default_rng(11)
    cm3 = engine.CostMatrix3(engine.CostMatrix.of_sub_indel(1, 2))
    ref = oracle.CM3(oracle.CM2.sub_indel(1, 2))
    L = engine.load()
    for k in range(16):
        anc = rand_seq(rng, int(rng.integers(0, 40)))
        s = [mutate(rng, anc, 0.15, 0.1) for _ in range(3)]
        if k == 0:
            s = [rand_seq(rng, 0), rand_seq(rng, 0), rand_seq(rng, 0)]
        if k == 1:
            s = [rand_seq(rng, 0), rand_seq(rng, 5), rand_seq(rng, 9)]
        cap = sum(len(x) for x in s) + 1
        outs = [np.zeros(cap, np.uint8) for _ in range(3)]
        ln = C.c_int32(0)
        cost = C.c_int32(0)
        rc = L.poyg_algn_align_3d(ctx.h, cm3.h, *[v for x in s for v in (engine._p8(x), len(x))],
                                  *[engine._p8(o) for o in outs], cap, C.byref(ln), C.byref(cost))
        assert rc == 0, engine.load().poyg_last_error()
        want = oracle.align_3(*s, ref)
        assert cost.value == want[0], k
        for o, w in zip(outs, want[1:]):
            assert np.array_equal(o[cap - ln.value:], w), k


def run_triples(ctx, cm2, T):
    """One triple plan over T (lists of three sequences): costs, aligned
    triples and medians as numpy arrays."""
    from poyd_amd import engine
    cm3 = engine.CostMatrix3(cm2)
    seqs = [x for t in T for x in t]
    bt = batch_of(seqs)
    off = bt.off.reshape(-1, 3)
    ln = bt.ln.reshape(-1, 3)
    plan = engine.TriplePlan(ctx, cm3, off[:, 0], ln[:, 0], off[:, 1], ln[:, 1], off[:, 2], ln[:, 2])
    d_seq = engine.DeviceBuffer.from_array(ctx, bt.seq)
    d_cost = engine.DeviceBuffer(ctx, 4 * len(T))
    d_out = engine.DeviceBuffer(ctx, plan.out_bytes)
    d_len = engine.DeviceBuffer(ctx, 16 * len(T))
    plan.run(d_seq.ptr, d_cost.ptr, d_out.ptr, d_len.ptr)
    ctx.sync()
    import ctypes as C
    bad = C.c_int32(0)
    engine.load().poyg_plan_status(plan.h, C.byref(bad))
    assert bad.value == 0
    cost = d_cost.download(np.int32, len(T))
    out = d_out.download(np.uint8, plan.out_bytes)
    lens = d_len.download(np.int32, 4 * len(T))
    res = []
    for k, t in enumerate(T):
        cap = ((sum(len(x) for x in t) + 1 + 15) // 16) * 16
        got = []
        for q in range(4):
            n = lens[4 * k + q]
            base = plan.out_off[k] + q * cap
            got.append(out[base + cap - n: base + cap].copy())
        res.append((int(cost[k]), got))
    plan.close()
    return res


def check_triples(ctx, oracle, sub, indel, T):
    from poyd_amd import engine
    cm2 = engine.CostMatrix.of_sub_indel(sub, indel)
    ref = oracle.CM3(oracle.CM2.sub_indel(sub, indel))
    got = run_triples(ctx, cm2, T)
    for k, t in enumerate(T):
        want = oracle.align_3(*t, ref)
        assert got[k][0] == want[0], (k, [len(x) for x in t])
        for q in range(3):
            assert np.array_equal(got[k][1][q], want[1 + q]), (k, q, [len(x) for x in t])
        assert np.array_equal(got[k][1][3], oracle.median_3(*want[1:], ref)), k


def test_three_d_batch_matches_oracle(ctx, oracle):
    note("three-dimensional batch")
    rng = np.random.default_rng(12)
    T = []
    for k in range(40):
        anc = rand_seq(rng, int(rng.integers(5, 60)))
        T.append([mutate(rng, anc, 0.15, 0.06) for _ in range(3)])
    check_triples(ctx, oracle, 1, 2, T)


def shaped_triples(rng, shapes):
    T = []
    for n1, n2, n3 in shapes:
        anc = rand_seq(rng, max(n1, n2, n3) - 1)
        t = []
        for n in (n1, n2, n3):
            x = mutate(rng, anc, 0.15, 0.04)[:n]
            if len(x) < n:
                x = np.concatenate([x, rand_seq(rng, n - len(x))[1:]]).astype(np.uint8)
            t.append(x)
        T.append(t)
    return T


# s3 lengths across every row width of the row kernel (64 * 4, 8, 12, 16
# cells) and past it (the chunked kernel), with degenerate planes and lines
CUBE_SHAPES = [(1, 1, 1), (1, 1, 9), (1, 7, 1), (6, 1, 1), (1, 5, 300), (4, 1, 520), (2, 2, 2),
               (9, 11, 255), (9, 11, 256), (9, 11, 257), (12, 8, 300), (7, 13, 511), (7, 13, 512),
               (7, 13, 513), (10, 9, 700), (5, 6, 768), (5, 6, 769), (6, 5, 1000), (4, 4, 1024),
               (3, 5, 1025), (4, 3, 1300), (40, 35, 90), (30, 45, 130)]


def test_three_d_row_classes(ctx, oracle):
    note("three-dimensional row classes, int16 rows")
    rng = np.random.default_rng(31)
    check_triples(ctx, oracle, 1, 2, shaped_triples(rng, CUBE_SHAPES))


# planes around the chunks' sizes (a plane p computes min(p + 1, 16) lines at a
# time; from plane 48 on the next chunk's inputs are loaded ahead), lines around
# multiples of 16, every row width
CHUNK_SHAPES = [(n1, n2, n3) for n1, n3 in ((15, 40), (17, 260), (47, 30), (48, 257), (49, 520), (50, 70), (66, 20))
                for n2 in (1, 2, 15, 16, 17, 33)] + [(97, 31, 300), (52, 32, 790), (49, 34, 512), (80, 70, 60),
                                                     (50, 16, 1000), (49, 47, 513), (60, 48, 256)]


@pytest.mark.parametrize("sub,indel", [(1, 2), (20, 30)])
def test_three_d_chunks(ctx, oracle, sub, indel):
    """The block kernels, packed (costs 1, 2) and not (20, 30)."""
    note(f"three-dimensional chunks, costs {sub} {indel}")
    rng = np.random.default_rng(33)
    check_triples(ctx, oracle, sub, indel, shaped_triples(rng, CHUNK_SHAPES if indel == 2 else CHUNK_SHAPES[::3]))


def test_three_d_wide_costs(ctx, oracle):
    note("three-dimensional row classes, int32 rows (costs past 2^15)")
    rng = np.random.default_rng(32)
    check_triples(ctx, oracle, 90, 200, shaped_triples(rng, CUBE_SHAPES[:18]))


# planes around the two-wave workgroup's chunks (min(p + 1, 4) lines; inputs ahead
# from plane 12 on), lines around multiples of 4, every row width
FEW_SHAPES = [(n1, n2, n3) for n1, n3 in ((1, 30), (2, 257), (4, 20), (5, 520), (12, 40), (13, 260), (14, 30), (17, 70))
              for n2 in (1, 2, 3, 4, 5, 8, 9)] + [(20, 21, 60), (26, 7, 300), (15, 12, 790), (13, 3, 1000), (16, 5, 512)]


@pytest.mark.parametrize("sub,indel,widest", [(1, 2, 512), (1, 2, 1024), (20, 30, 1024), (90, 200, 1024)])
def test_three_d_many_small(ctx, oracle, sub, indel, widest):
    """Batches of small triples, which take workgroups of two waves: packed
    (costs 1, 2; rows of at most 512 cells and wider ones), 16-bit and 32-bit
    rows."""
    note(f"three-dimensional small triples, costs {sub} {indel}")
    from poyd_amd import engine
    rng = np.random.default_rng(38)
    shapes = [s for s in FEW_SHAPES if s[2] <= widest]
    some = shaped_triples(rng, shapes)
    pick = np.concatenate([np.arange(len(some)), np.repeat(np.arange(len(some)), 140)])
    got = run_triples(ctx, engine.CostMatrix.of_sub_indel(sub, indel), [some[k] for k in pick])
    ref = oracle.CM3(oracle.CM2.sub_indel(sub, indel))
    want = [oracle.align_3(*t, ref) for t in some]
    med = [oracle.median_3(*w[1:], ref) for w in want]
    for q, k in enumerate(pick):
        assert got[q][0] == want[k][0], (q, shapes[k])
        assert all(np.array_equal(got[q][1][x], want[k][1 + x]) for x in range(3)), (q, shapes[k])
        assert np.array_equal(got[q][1][3], med[k]), (q, shapes[k])


@pytest.mark.parametrize("sub,indel", [(1, 2), (20, 30)])
def test_three_d_more_long_rows_than_waves(ctx, oracle, sub, indel):
    """Rows above 1,024 cells, more triples than the chunked kernel has waves
    (2,048), with every row width of the block kernels beside them."""
    from poyd_amd import engine
    note(f"three-dimensional long rows, costs {sub} {indel}")
    rng = np.random.default_rng(37)
    some = shaped_triples(rng, [(n1, n2, n3) for n1, n2 in ((2, 3), (4, 2), (3, 3)) for n3 in (1025, 1030, 1089)] +
                          [(3, 4, 200), (4, 3, 500), (5, 2, 700), (2, 2, 1000)])
    pick = np.concatenate([np.arange(len(some)), rng.integers(0, 9, 2300)])
    got = run_triples(ctx, engine.CostMatrix.of_sub_indel(sub, indel), [some[k] for k in pick])
    ref = oracle.CM3(oracle.CM2.sub_indel(sub, indel))
    want = [oracle.align_3(*t, ref) for t in some]
    for q, k in enumerate(pick):
        assert got[q][0] == want[k][0], (q, k)
        assert all(np.array_equal(got[q][1][x], want[k][1 + x]) for x in range(3)), (q, k)


def test_fitch_matches_oracle(ctx, oracle):
    from poyd_amd import engine
    note("fitch down/up")
    rng = np.random.default_rng(13)
    for length in (1, 17, 10000, 4096):
        a, b, c, d = (rng.integers(1, 256, length).astype(np.uint8) for _ in range(4))
        res = np.zeros(length, np.uint8)
        import ctypes as C
        added = C.c_int64(0)
        L = engine.load()
        assert L.poyg_nonadd_median(ctx.h, engine._p8(a), engine._p8(b), engine._p8(res), length, C.byref(added)) == 0
        want, wadd = oracle.nonadd_median(a, b)
        assert np.array_equal(res, want) and added.value == wadd
        assert L.poyg_nonadd_median_3(ctx.h, engine._p8(a), engine._p8(b), engine._p8(c), engine._p8(d),
                                      engine._p8(res), length) == 0
        assert np.array_equal(res, oracle.nonadd_median_3(a, b, c, d))


def test_fitch_host_batches_match_oracle(ctx, oracle):
    """poyg_fitch_pairs_host (engine.fitch_pairs): batches of row pairs over
    host arrays, every median row and change count equal to the oracle's
    nonadd_median, for odd lengths, one row and many, and an empty batch."""
    from poyd_amd import engine
    note("fitch host batches")
    rng = np.random.default_rng(14)
    for n, length in ((1, 1), (3, 17), (40, 1001), (700, 64), (5, 10000)):
        a = rng.integers(1, 256, (n, length)).astype(np.uint8)
        b = rng.integers(1, 256, (n, length)).astype(np.uint8)
        b[:, ::3] = a[:, ::3]   # some characters agree
        res, added = engine.fitch_pairs(ctx, a, b)
        for k in range(n):
            want, wadd = oracle.nonadd_median(a[k], b[k])
            assert np.array_equal(res[k], want) and int(added[k]) == wadd, (n, length, k)
    res, added = engine.fitch_pairs(ctx, np.zeros((0, 8), np.uint8), np.zeros((0, 8), np.uint8))
    assert res.shape == (0, 8) and added.shape == (0,)


def test_workload_pairwise_linear_1000(ctx, oracle):
    """The 1,000-pair linear workload (L 200-400, 10% subs, 2% indels),
    every pair bit-exact: cost, both aligned sequences and the median."""
    from poyd_amd import engine
    note("workload pairwise-linear-1000")
    w = synth.workload_linear_1000()
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    ref = oracle.CM2.sub_indel(1, 2)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_ALIGN, w.a, w.b)
    for k in range(len(w.a)):
        a, b = w.a.get(k), w.b.get(k)
        cost, oa, ob = oracle.align_2(a, b, ref)
        assert res.cost[k] == cost
        assert np.array_equal(res.seq(k, 0), oa) and np.array_equal(res.seq(k, 1), ob)
        assert np.array_equal(res.seq(k, 2), oracle.median_2(oa, ob, ref))


def test_workload_pairwise_affine_sample(ctx, oracle):
    """The 65,536-pair affine workload: a seeded sample of 1,500 pairs
    bit-exact (all four outputs and the cost) and, for all pairs, the
    size-independent properties: recost of the alignment equals the cost and
    stripping gaps returns the inputs."""
    from poyd_amd import engine
    note("workload pairwise-affine-65536")
    w = synth.workload_affine_65536()
    cm = engine.CostMatrix.of_sub_indel(1, 1, 3)
    ref = oracle.CM2.sub_indel(1, 1, 3)
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_AFFINE_ALIGN, w.a, w.b)
    rng = np.random.default_rng(5)
    sample = rng.choice(len(w.a), size=1500, replace=False)
    for k in sample:
        a, b = w.a.get(k), w.b.get(k)
        med, ri, rj, cost, mwg = oracle.align_affine_3(a, b, ref)
        assert res.cost[k] == cost, k
        for slot, want in enumerate((med, mwg, ri, rj)):
            assert np.array_equal(res.seq(k, slot), want), (k, slot)
    bad = 0
    for k in range(len(w.a)):
        ri, rj = res.seq(k, 2), res.seq(k, 3)
        if oracle.verify_2(ri, rj, ref) != res.cost[k]:
            bad += 1
        elif not (np.array_equal(ri[ri != GAP], w.a.get(k)[1:]) and np.array_equal(rj[rj != GAP], w.b.get(k)[1:])):
            bad += 1
    assert bad == 0


@pytest.mark.parametrize("mm,go,ge", [(1, 2, 1), (2, 0, 1), (1, 3, 2)])
def test_powell_matches_oracle(ctx, oracle, mm, go, ge):
    from poyd_amd import engine
    note(f"powell_3d mm={mm} go={go} ge={ge}")
    rng = np.random.default_rng(50 + mm + 7 * go + 13 * ge)
    shapes = [(0, 0, 0), (0, 3, 5), (4, 0, 0), (1, 1, 1), (7, 7, 7)] + \
             [tuple(int(v) for v in rng.integers(1, 60, size=3)) for _ in range(12)] + [(150, 140, 160)]
    for n1, n2, n3 in shapes:
        anc = rand_seq(rng, max(n1, n2, n3, 1))
        t = []
        for n in (n1, n2, n3):
            x = mutate(rng, anc, 0.15, 0.05)[:n + 1]
            if len(x) < n + 1:
                x = np.concatenate([x, rand_seq(rng, n + 1 - len(x))[1:]]).astype(np.uint8)
            t.append(x)
        cost, al = engine.powell_3d(ctx, *t, mm, go, ge)
        # the reference's own search picks the alignment (its cost is the
        # model's least cost, except that three equal strings cost 1: the
        # search's loop starts at cost 1)
        want = oracle.powell_ukk(*t, mm, go, ge)
        least = oracle.powell_3d(*t, mm, go, ge)[0]
        same = all(len(x) == len(t[0]) and np.array_equal(x, t[0]) for x in t)
        assert cost == want[0] == (1 if same else least), (n1, n2, n3)
        for q in range(3):
            assert np.array_equal(al[q], want[1 + q]), (n1, n2, n3, q)


def test_powell_search_choices(ctx, oracle):
    # divergent triples, where least-cost alignments are many and the
    # check-point recursion runs several levels deep: the engine's alignment
    # is the reference search's, column for column
    from poyd_amd import engine
    note("powell_3d search choices")
    rng = np.random.default_rng(58)
    for k in range(8):
        mm, go, ge = [(1, 2, 1), (2, 0, 1), (1, 3, 2), (3, 1, 1), (1, 3, 1)][k % 5]
        anc = rand_seq(rng, int(rng.integers(40, 100)))
        t = [mutate(rng, anc, 0.3, 0.1) for _ in range(3)]
        cost, al = engine.powell_3d(ctx, *t, mm, go, ge)
        want = oracle.powell_ukk(*t, mm, go, ge)
        assert cost == want[0] == oracle.powell_3d(*t, mm, go, ge)[0], k
        for q in range(3):
            assert np.array_equal(al[q], want[1 + q]), (k, q)


@pytest.mark.parametrize("mm,go,ge", [(1, 2, 1), (3, 4, 2), (2, 1, 3)])
def test_powell_run_lengths(ctx, oracle, mm, go, ge):
    """Runs of equal characters around a row's sixteen columns, up to the ends
    of the sequences, and levels whose diagonals fill the last workgroup by
    one to all of its sixteen rows (the boxes grow by odd squares)."""
    from poyd_amd import engine
    note(f"powell_3d run lengths mm={mm} go={go} ge={ge}")
    rng = np.random.default_rng(61 + mm + 7 * go + 13 * ge)
    for run in (15, 16, 17, 31, 32, 33, 49):
        a = rand_seq(rng, 3 * run)
        b, c = a.copy(), a.copy()
        b[1 + run] = 1 if b[1 + run] != 1 else 2          # one substitution after the first run
        c = np.delete(c, 1 + 2 * run)                     # one gap after the second
        c = c[:len(c) - (run % 3)]                        # and ends of unequal length
        for t in ([a, b, c], [c, a, b]):
            cost, al = engine.powell_3d(ctx, *t, mm, go, ge)
            want = oracle.powell_ukk(*t, mm, go, ge)
            assert cost == want[0], run
            for q in range(3):
                assert np.array_equal(al[q], want[1 + q]), (run, q)


def test_powell_rejects_gap_only_characters(ctx):
    from poyd_amd import engine
    x = np.array([16, 1, 16, 2], np.uint8)
    with pytest.raises(engine.PoygError):
        engine.powell_3d(ctx, x, x, x, 1, 2, 1)


def test_device_cache_reuse(ctx):
    """Blocks released to the per-device cache come back only after a
    synchronization, and a reused block holds what its new owner wrote."""
    from poyd_amd import engine
    note("device cache reuse")
    rng = np.random.default_rng(5)
    live = []
    for cycle in range(40):
        size = int(rng.choice([100, 256, 4000, 70000, 1 << 20]))
        data = rng.integers(0, 256, size, dtype=np.uint8)
        b = engine.DeviceBuffer.from_array(ctx, data)
        live.append((b, data))
        if cycle % 3 == 2:
            # release one buffer without a sync: a block allocated now must not be it
            old, _ = live.pop(0)
            ptr = old.ptr
            old.free()
            fresh = engine.DeviceBuffer(ctx, 16)
            assert fresh.ptr != ptr
            fresh.free()
        if cycle % 7 == 6:
            ctx.sync()
        for b2, d2 in live:
            assert np.array_equal(b2.download(np.uint8, len(d2)), d2), cycle
    for b2, _ in live:
        b2.free()
    ctx.sync()


def test_linear_fill_wait_gives_up_reported(ctx, oracle, monkeypatch):
    """The systolic fill's wait for the previous strip of a pair is a bounded
    poll.  With the poll limit forced to zero from the host, the waits give
    up at once: the kernel still ends, the plan reports the pairs as failed
    and the engine raises; the next run with the default limit is exact."""
    from poyd_amd import engine
    note("linear fill wait gives up")
    rng = np.random.default_rng(17)
    A = [rand_seq(rng, 1500) for _ in range(4)]
    B = [mutate(rng, a, 0.1, 0.03) for a in A]
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    ref = oracle.CM2.sub_indel(1, 2)
    monkeypatch.setenv("POYG_SYS_SPIN_LIMIT", "0")
    # these pairs would go to the packed fill, which has no waits: the
    # systolic fill takes them here
    ctx.set_tuning("lin_cost_kernel", 1)
    try:
        # each failed pair counts once, however many of its waves gave up
        with pytest.raises(engine.PoygError, match=r"\b[1-4] pairs failed"):
            engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_ALIGN, batch_of(A), batch_of(B))
    finally:
        ctx.set_tuning("lin_cost_kernel", -1)
    monkeypatch.delenv("POYG_SYS_SPIN_LIMIT")
    res = engine.run_pairs(ctx, cm, engine.POYG_MODE_LINEAR_ALIGN, batch_of(A), batch_of(B))
    for k, (a, b) in enumerate(zip(A, B)):
        cost, oa, ob = oracle.align_2(a, b, ref)
        assert res.cost[k] == cost, k
        assert np.array_equal(res.seq(k, 0), oa), k


def test_plan_rejects_what_the_kernels_cannot_hold(ctx):
    """Planning refuses, before any allocation or launch: a linear matrix
    with a negative entry (POYG_EINVAL: the kernels' out-of-band marker must
    stay above every cell value), and a linear alignment whose direction band
    reaches the kernels' 32-bit offsets (POYG_EUNSUPPORTED)."""
    import ctypes as C
    from poyd_amd import engine
    note("plan guards")
    L = engine.load()
    cm = engine.CostMatrix.of_sub_indel(1, 2)
    neg = engine.CostMatrix.of_list([[0, -1, 1, 1, 2], [-1, 0, 1, 1, 2], [1, 1, 0, 1, 2], [1, 1, 1, 0, 2],
                                     [2, 2, 2, 2, 0]])

    def plan(m, mode, la, lb, dw):
        h = C.c_void_p()
        rc = L.poyg_plan_pairs(ctx.h, m.h, mode, 1, (C.c_int64 * 1)(0), (C.c_int32 * 1)(la),
                               (C.c_int64 * 1)(0), (C.c_int32 * 1)(lb), (C.c_int32 * 1)(dw), C.byref(h))
        if rc == 0:
            L.poyg_plan_destroy(h)
        return rc

    assert plan(cm, engine.POYG_MODE_LINEAR_ALIGN, 300, 280, 40) == 0
    assert plan(neg, engine.POYG_MODE_LINEAR_COST, 300, 280, 40) == -1
    assert plan(cm, engine.POYG_MODE_LINEAR_ALIGN, 60000, 40000, 100) == -4
    assert plan(cm, engine.POYG_MODE_LINEAR_COST, 60000, 40000, 100) == 0   # no direction band


@pytest.mark.parametrize("width", [1, 2, 4])
def test_fitch_widths_match_oracle(ctx, oracle, width):
    """NonaddCS8/16/32: the down and up passes at 1, 2 and 4 bytes per
    character, with state sets over every bit of the width, row lengths
    that are and are not multiples of 16 bytes."""
    import ctypes as C
    from poyd_amd import engine
    note(f"fitch width {width}")
    dt = {1: np.uint8, 2: np.uint16, 4: np.uint32}[width]
    rng = np.random.default_rng(40 + width)
    L = engine.load()
    for length in (1, 7, 1000, 4096, 10003):
        a, b, c, d = (rng.integers(1, 1 << (8 * width), size=length, dtype=np.uint64).astype(dt) for _ in range(4))
        # sparse sets too, so that empty intersections occur at every width
        a[::3] = (np.uint64(1) << rng.integers(0, 8 * width, size=len(a[::3])).astype(np.uint64)).astype(dt)
        b[::3] = (np.uint64(1) << rng.integers(0, 8 * width, size=len(b[::3])).astype(np.uint64)).astype(dt)
        res = np.zeros(length, dt)
        added = C.c_int64(0)
        assert L.poyg_nonadd_median_w(ctx.h, width, a.ctypes.data, b.ctypes.data, res.ctypes.data, length,
                                      C.byref(added)) == 0
        want, wadd = oracle.nonadd_median_w(a, b, width)
        assert np.array_equal(res, want) and added.value == wadd, length
        assert L.poyg_nonadd_median_3_w(ctx.h, width, a.ctypes.data, b.ctypes.data, c.ctypes.data, d.ctypes.data,
                                        res.ctypes.data, length) == 0
        assert np.array_equal(res, oracle.nonadd_median_3_w(a, b, c, d, width)), length


@pytest.mark.parametrize("width", [1, 2, 4])
def test_fitch_ragged_levels(ctx, oracle, width):
    """A level of several nodes whose rows start at any byte: row lengths
    around the 16-byte vectors and the workgroups' share, the result written
    over an input too, the bytes before and after the rows left alone."""
    import ctypes as C
    from poyd_amd import engine
    dt = {1: np.uint8, 2: np.uint16, 4: np.uint32}[width]
    rng = np.random.default_rng(90 + width)
    L = engine.load()
    for length in (1, 3, 15, 16, 17, 31, 4095, 4097, 65537):
        note(f"fitch level width {width} length {length}")
        rows = (np.uint64(1) << rng.integers(0, 8 * width, size=(9, length)).astype(np.uint64)).astype(dt)
        rows |= (rng.random((9, length)) < 0.3) * (np.uint64(1) << rng.integers(0, 8 * width, size=(9, length)).astype(
            np.uint64)).astype(dt)
        host = np.concatenate([np.full(3, 7, dt), rows.ravel(), np.full(5, 9, dt)])
        d = engine.DeviceBuffer.from_array(ctx, host)
        at = d.ptr + 3 * width
        jobs = np.array([[0, 1, 4], [2, 3, 5], [6, 7, 7]], np.int32)   # the last one in place
        d_jobs = engine.DeviceBuffer.from_array(ctx, np.ascontiguousarray(jobs.T))
        d_added = engine.DeviceBuffer.from_array(ctx, np.zeros(3, np.int64))
        assert L.poyg_fitch_down_w(ctx.h, width, at, length, 3, d_jobs.ptr, d_jobs.ptr + 12, d_jobs.ptr + 24,
                                   d_added.ptr, None) == 0
        ctx.sync()
        got = d.download(dt, len(host))
        added = d_added.download(np.int64, 3)
        want = rows.copy()
        for k, (a, b, r) in enumerate(jobs):
            want[r], n = oracle.nonadd_median_w(rows[a], rows[b], width)
            assert added[k] == n, (length, k)
        assert np.array_equal(got[3:-5].reshape(9, length), want), length
        up = np.array([[8, 4, 0, 1, 6], [8, 5, 2, 3, 5]], np.int32)
        d_up = engine.DeviceBuffer.from_array(ctx, np.ascontiguousarray(up.T))
        assert L.poyg_fitch_up_w(ctx.h, width, at, length, 2, *[d_up.ptr + 8 * c for c in range(5)], None) == 0
        ctx.sync()
        got = d.download(dt, len(host))
        final = want.copy()
        for A, N, D1, D2, F in up:
            final[F] = oracle.nonadd_median_3_w(want[A], want[N], want[D1], want[D2], width)
        assert np.array_equal(got[3:-5].reshape(9, length), final), length
        assert (got[:3] == 7).all() and (got[-5:] == 9).all()
