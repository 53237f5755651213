"""The packed one-workgroup substitution's cases: every number of chunks (4
entries) summed ahead of a group's barrier (0 to 4) with every number behind
it (0 to 6 in registers, and more from memory), rows of every remainder modulo
4, slices of 1 to 64 rows, level sets of one slice, several and more than 12;
the factors that the form refuses (a row of more than 1000 entries, a
dependency that lies further back than the window) beside those that it just
takes.  The path is read back in every case, and values are bit for bit those
of the sequential substitution, in FP64 and FP32."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


WAVES, AHEAD, BEHIND = 12, 4, 6


def plan(irp, ja, level):
    """(chunks ahead, chunks behind, rows) of every slice: level sets in order, the longest rows first, 64 rows to a
    slice, WAVES slices to a group; ahead: leading chunks without a row of the group before."""
    n, ln = level.size, np.diff(irp)
    order = np.lexsort((np.arange(n), -ln, level))
    pos = np.empty(n, int)
    pos[order] = np.arange(n)
    group, g, out = np.empty(n, int), -1, []
    for lv in range(level.max() + 1):
        rows = order[level[order] == lv]
        for s in range(0, rows.size, 64):
            if s // 64 % WAVES == 0:
                g += 1
            sl = rows[s:s + 64]
            group[pos[sl]] = g
            nc = -(-ln[sl[0]] // 4)
            ke = min(nc, AHEAD)
            for r in sl:
                gg = group[pos[ja[irp[r]:irp[r] + min(4 * ke, ln[r])]]]
                near = np.nonzero(gg >= g - 1)[0]
                if near.size:
                    ke = near[0] // 4
            out.append((ke, nc - ke, sl.size))
    return out


def factor(upper, seed):
    """A strict triangle whose level sets run through all pairs of chunks ahead and behind.  Two regions: chain rows
    (C: 32 a level set, each on a row of the level set before) and work rows (W: on W rows two and more level sets
    back, the first 4 ke entries, then on C rows of the level set before).  In a row W columns come first: C is
    numbered behind W in an upper triangle, and level set by level set in a lower one."""
    rng = np.random.default_rng(seed)
    want = [(0, 1)] * 3 + [(ke, lt) for ke in range(AHEAD + 1) for lt in range(1, BEHIND + 3)] + [(4, 1), (0, 8)]
    sizes = [int(rng.choice([64, 65, 96, 97, 128, 150])) for _ in want]  # (whole slices of work rows first)
    for q in (9, 21, 34):
        sizes[q] = 800  # more slices than wavefronts: two groups in a level set
    nlev, C = len(want) + 1, 32
    wrows, crows, nxt = [np.zeros(0, int)], [], 0
    if not upper:
        ids = []
        for lv in range(nlev):
            m = 0 if lv == 0 else sizes[lv - 1]
            ids.append((nxt + np.arange(m), nxt + m + np.arange(C)))
            nxt += m + C
        wrows, crows = [i[0] for i in ids], [i[1] for i in ids]
    else:
        nw = sum(sizes)
        at = nw
        for lv in range(1, nlev):  # later level sets in front
            at -= sizes[lv - 1]
            wrows.append(at + np.arange(sizes[lv - 1]))
        crows = [nw + (nlev - 1 - lv) * C + np.arange(C) for lv in range(nlev)]
        nxt = nw + nlev * C
    n = nxt
    level, cols = np.zeros(n, int), [None] * n
    for lv in range(nlev):
        for r in crows[lv]:
            level[r] = lv
            cols[r] = np.zeros(0, int) if lv == 0 else np.array([rng.choice(crows[lv - 1])])
        for k, r in enumerate(wrows[lv]):
            level[r] = lv
            ke, lt = want[lv - 1]
            back = np.concatenate([wrows[q] for q in range(1, lv - 1)] + [np.zeros(0, int)])
            if not upper:  # C rows of old level sets serve too
                back = np.concatenate([back] + [crows[q] for q in range(max(0, lv - 1))])
            early = np.sort(rng.choice(back, 4 * ke, replace=False)) if back.size >= 4 * ke else np.zeros(0, int)
            late = np.sort(rng.choice(crows[lv - 1], 4 * lt - int(rng.integers(0, 4)) * (k > 0), replace=False))
            cols[r] = np.concatenate([early, late])
            assert (np.diff(cols[r]) > 0).all()
    irp = np.concatenate([[0], np.cumsum([c.size for c in cols])])
    ja = np.concatenate(cols)
    return irp, ja, rng.uniform(-0.2, 0.2, ja.size), level


def sequential(irp, ja, val, level, b, d, kind, V):
    """kind 0: t = b - acc; 1: d b - acc; 2: (b - acc) / d; products added in stored order, rounded to V."""
    t = [V(0)] * level.size
    val, b, d = [V(v) for v in val], [V(v) for v in b], [V(v) for v in d]
    irp, ja = irp.tolist(), ja.tolist()
    for r in np.argsort(level, kind="stable").tolist():
        acc = V(0)
        for k in range(irp[r], irp[r + 1]):
            acc = acc + val[k] * t[ja[k]]
        t[r] = d[r] * b[r] - acc if kind == 1 else ((b[r] - acc) / d[r] if kind == 2 else b[r] - acc)
    return np.array(t, dtype=V)


def handle(eng, solver, n, dv, lower, upper, precision="double"):
    p = eng.MldPrec(device=0).init("BJAC" if solver == "ILU" else "GS")
    p.set_precision(precision)
    p.upload_level(0, sp.identity(n, format="csr"))
    none = (np.zeros(n + 1, np.int64), np.zeros(0, np.int32), np.zeros(0))
    tri = [none if t is None else t[:3] for t in (lower, upper)]
    p.upload_smoother(0, solver, dv=dv, l=tri[0], u=tri[1])
    return p.finalize_hierarchy(1)


def packed(err):
    return "packed for one workgroup" in err


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("solver", ["ILU", "GS"])
def test_cases(eng, monkeypatch, capfd, solver, precision):
    monkeypatch.setenv("MLD_VERBOSE", "1")
    L = factor(False, 1)
    U = factor(True, 2)
    pl, pu = plan(L[0], L[1], L[3]), plan(U[0], U[1], U[3])
    for pairs, name in ((pl, "L"), (pu, "U")):
        seen = {(k, min(b, BEHIND + 1)) for k, b, _ in pairs}
        assert {(k, b) for k in range(AHEAD + 1) for b in range(1, BEHIND + 2)} <= seen, name
        assert {1, 64} <= {m for _, _, m in pairs}
    n = L[0].size - 1
    V = float if precision == "double" else np.float32
    n = max(n, U[0].size - 1)  # both of one size: unknowns without entries at the end
    pad = lambda f: (np.concatenate([f[0], np.full(n + 1 - f[0].size, f[0][-1])]), f[1], f[2],  # noqa: E731
                     np.concatenate([f[3], np.zeros(n + 1 - f[0].size, int)]))
    L, U = pad(L), pad(U)
    rng = np.random.default_rng(5)
    dv = rng.uniform(0.5, 2.0, n)
    x = rng.standard_normal(n)
    if precision == "mixed":
        x = x.astype(np.float32).astype(np.float64)
    capfd.readouterr()
    p = handle(eng, solver, n, dv, L, U if solver == "ILU" else None, precision)
    assert packed(capfd.readouterr().err)
    if solver == "ILU":
        t = sequential(*L, x, dv, 0, V)
        ref = sequential(*U, t, dv, 1, V)
    else:
        ref = sequential(*L, x, dv, 2, V)
    for turn in range(3):
        y = p.apply(dev(x)).cpu().numpy()
        assert (y == ref.astype(np.float64)).all(), turn


def chain(n, far, longest, seed):
    """Lower triangle: row r on row r - 1, row `far` + 200 also on row 200, and one row of `longest` entries."""
    rng = np.random.default_rng(seed)
    cols = [np.array([r - 1]) if r else np.zeros(0, int) for r in range(n)]
    if far:
        cols[far + 200] = np.array([200, far + 199])
    if longest:
        cols[longest + 50] = np.arange(50, longest + 50)
    irp = np.concatenate([[0], np.cumsum([c.size for c in cols])])
    ja = np.concatenate(cols)
    return irp, ja, rng.uniform(-0.2, 0.2, ja.size), np.arange(n)


# the window holds (163840 - 64) / 8 = 20472 rows in FP64, 32766 in FP32
@pytest.mark.parametrize("precision,far,longest,taken", [
    ("double", 20471, 0, True), ("double", 20472, 0, False), ("mixed", 32765, 0, True), ("mixed", 32766, 0, False),
    ("double", 0, 1000, True), ("double", 0, 1001, False), ("mixed", 0, 997, True)])
def test_refusals(eng, monkeypatch, capfd, precision, far, longest, taken):
    print(f"[packed refusals] {precision} far {far} longest {longest}", flush=True)
    monkeypatch.setenv("MLD_VERBOSE", "1")
    n = far + 700 if far else 3000
    L = chain(n, far, longest, n)
    rng = np.random.default_rng(n)
    dv = rng.uniform(0.5, 2.0, n)
    x = rng.standard_normal(n).astype(np.float32).astype(np.float64)
    capfd.readouterr()
    p = handle(eng, "GS", n, dv, L, None, precision)
    assert packed(capfd.readouterr().err) == taken
    ref = sequential(*L, x, dv, 2, float if precision == "double" else np.float32)
    assert (p.apply(dev(x)).cpu().numpy() == ref.astype(np.float64)).all()
