"""Graph capture: applications are launches alone and replay with the eager
result, whatever packed form they take; what reads scalars on the host (solves,
K-cycles) is refused, and the handle works as before afterwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def build(eng, A, smoother, cycle, precision):
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 2 if "JACOBI" in smoother else 1),
                 ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 100),
                 ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
        p.set(k, v)
    return p.set_precision(precision).build(A)


@pytest.mark.parametrize("smoother,cycle,precision", [
    ("L1-JACOBI", "VCYCLE", "double"), ("L1-JACOBI", "WCYCLE", "mixed"), ("FBGS", "VCYCLE", "double"),
    ("BJAC", "VCYCLE", "double")])
def test_replays(eng, orc, smoother, cycle, precision):
    print(f"[capture] {smoother} {cycle} {precision}", flush=True)
    A = orc.gen_pde3d(64).to_scipy()
    n = A.shape[0]
    p = build(eng, A, smoother, cycle, precision)
    rng = np.random.default_rng(3)
    x = torch.from_numpy(rng.standard_normal(n)).to("cuda:0")
    y = torch.empty_like(x)
    z = torch.empty_like(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        p.apply(x, y)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        p.apply(x, y)
    for turn in range(4):
        x.copy_(torch.from_numpy(rng.standard_normal(n)))
        g.replay()
        torch.cuda.synchronize()
        p.apply(x, z)  # the program's own work between the replays
        torch.cuda.synchronize()
        assert torch.equal(y, z), turn


@pytest.mark.parametrize("what", ["CG", "FCG", "BICGSTAB", "apply"])
def test_refused(eng, orc, what):
    A = orc.gen_pde3d(24).to_scipy()
    n = A.shape[0]
    p = build(eng, A, "L1-JACOBI", "KCYCLESYM" if what == "apply" else "VCYCLE", "double")
    x = torch.from_numpy(np.random.default_rng(4).standard_normal(n)).to("cuda:0")
    y = torch.empty_like(x)

    def call():
        if what == "apply":
            return p.apply(x, y).clone()
        return eng.psb_krylov(what, A, p, x, torch.zeros_like(x), eps=1e-8)[0]

    before = call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with pytest.raises(eng.MldError, match="graph capture"):
        with torch.cuda.graph(g):
            if what == "apply":
                p.apply(x, y)
            else:
                eng.psb_krylov(what, A, p, x, y, eps=1e-8)
    torch.cuda.synchronize()
    for _ in range(2):
        assert torch.equal(call(), before)


@pytest.mark.parametrize("method", ["CG", "FCG"])
def test_solve_beside_a_capture(eng, orc, method):
    """A solve on its own stream while another is captured in relaxed mode (the
    other modes forbid waiting on any stream meanwhile): accepted."""
    A = orc.gen_pde3d(64).to_scipy()
    n = A.shape[0]
    p = build(eng, A, "L1-JACOBI", "VCYCLE", "double")
    rng = np.random.default_rng(5)
    b = torch.from_numpy(rng.standard_normal(n)).to("cuda:0")
    x = torch.zeros_like(b)
    v = torch.from_numpy(rng.standard_normal(n)).to("cuda:0")
    v0 = v.clone()
    captured, own = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(own):
        want = eng.psb_krylov(method, A, p, b, torch.zeros_like(b), eps=1e-8)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(captured):
        g.capture_begin(capture_error_mode="relaxed")
        try:
            v.mul_(2.0)
            with torch.cuda.stream(own):
                got = eng.psb_krylov(method, A, p, b, x, eps=1e-8)
        finally:
            g.capture_end()
    torch.cuda.synchronize()
    assert got[1:] == want[1:] and torch.equal(got[0], want[0])
    for turn in range(1, 4):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(v, v0 * 2.0 ** turn)
