"""Adjoint solves whose transpose is stored in another layout than A: A has
rows of one length (ELL, one lane per row), A^T rows of very uneven ones
(several lanes per row), so that the dots of its products have more partial
sums than those of A.  The residual that a solve reports has to be that of its
solution, in every method and precision, also where the scalars and tickets
that lie behind the partial sums are used again by a further solve."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def uniform_rows(n, w, seed):
    """n x n, w entries in every row: a large diagonal, one of the first 64
    columns, and w - 2 others near the diagonal."""
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    cols = [i, rng.integers(0, 64, n)]
    for k in range(1, w - 1):
        cols.append((i + 64 + 97 * k + rng.integers(0, 97, n)) % n)
    cols = np.stack(cols, 1)
    for k in range(1, w):  # distinct columns in every row
        while True:
            same = (cols[:, k:k + 1] == cols[:, :k]).any(1)
            if not same.any():
                break
            cols[same, k] = (cols[same, k] + 1) % n
    vals = rng.uniform(-4.0, 4.0, (n, w)) / n ** 0.5
    vals[:, 0] = 4.0 + rng.uniform(0.0, 1.0, n)
    a = sp.csr_matrix((vals.reshape(-1), (np.repeat(i, w), cols.reshape(-1))), shape=(n, n))
    a.sort_indices()
    return a


@pytest.mark.parametrize("n,w", [(3800, 8), (4096, 16), (20000, 12), (32000, 16), (32767, 9)])
@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_adjoint(eng, n, w, precision):
    print(f"[adjoint layouts] n {n} w {w} {precision}", flush=True)
    A = uniform_rows(n, w, n + w)
    assert (np.diff(A.indptr) == w).all() and np.diff(A.tocsc().indptr).max() > 64
    b = np.random.default_rng(n).standard_normal(n)
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", 2)
    p.set_precision(precision).build(A)
    assert p.op_format(0, "A")["fmt"] == "ELL"
    first = {}
    for turn in range(2):
        for method in ("CG", "FCG", "BICGSTAB"):
            x, it, err = eng.psb_krylov_adjoint(method, p, dev(b), eps=1e-10)
            x = x.cpu().numpy()
            r = np.linalg.norm(b - A.T @ x) / np.linalg.norm(b)
            # the recursive residual and the true one part by the rounding of the products
            assert 0 < it < 100 and err <= 1e-10 and abs(r - err) <= 1e-13 * (4 + it), (method, it, err, r)
            if turn == 0:
                first[method] = x
            else:
                assert (x == first[method]).all(), method
        x, it, err = eng.psb_krylov("BICGSTAB", A, p, dev(b), eps=1e-10)
        r = np.linalg.norm(b - A @ x.cpu().numpy()) / np.linalg.norm(b)
        assert err <= 1e-10 and abs(r - err) <= 1e-13 * (4 + it)


def test_adjoint_multilevel(eng):
    """The dot of the fine level's last sweep with ND^T in such a layout."""
    n, w = 20000, 10
    A = uniform_rows(n, w, 3)
    b = np.random.default_rng(4).standard_normal(n)
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", "JACOBI"), ("SMOOTHER_SWEEPS", 2), ("AGGR_PROL", "SMOOTHED"), ("AGGR_THRESH", 0.0),
                 ("MIN_COARSE_SIZE", 200), ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU")):
        p.set(k, v)
    p.build(A)
    for method in ("CG", "FCG"):
        x, it, err = eng.psb_krylov_adjoint(method, p, dev(b), eps=1e-10)
        r = np.linalg.norm(b - A.T @ x.cpu().numpy()) / np.linalg.norm(b)
        assert 0 < it < 100 and err <= 1e-10 and abs(r - err) <= 1e-13 * (4 + it), (method, it, err, r)
