"""GPU: the reported plan of a batch of few short instances is the launched one
(a workgroup per instance, one split candidate to tune), and an instance that
became inactive leaves the others' results as they are on the bins."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _solver(pkg, horizons):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    s = pkg.Solver(pkg.default_config(max_knots=max(horizons), max_instances=len(horizons),
                                      max_total_knots=int(sum(horizons))))
    s.batch_setup(horizons)
    return s


def test_layout_and_autotune(pkg):
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count if torch.cuda.is_available() else 0
    short = [8] * (2 * n_cu)
    s = _solver(pkg, short)
    try:
        for items in (8, 2):
            s.batch_set_plan(split=1, max_items=items)
            assert s.batch_pcg_layout()["bins"] == len(short)
        assert sum(r["split"] for r in s.batch_autotune(iters=4, reps=1)) == 1
    finally:
        s.close()
    s = _solver(pkg, short + [65])  # on shared bins
    try:
        assert s.batch_pcg_layout()["bins"] < len(short)
        assert sum(r["split"] for r in s.batch_autotune(iters=4, reps=1)) == 3
    finally:
        s.close()


def test_inactive_instances(pkg):
    horizons, dead = [2, 17, 64, 5, 33, 16, 48], (1, 4)
    out = []
    for extra in ([], [65]):  # the short kernel, the bins
        h = horizons + extra
        g = [torch.Generator().manual_seed(300 + N) for N in h]
        xu = torch.cat([0.3 * torch.randn(21 * N - 7, generator=q) for N, q in zip(h, g)]).cuda()
        lam = torch.cat([0.01 * torch.randn(14 * N, generator=q) for N, q in zip(h, g)]).cuda()
        ees = [torch.rand(6 * N, generator=q) for N, q in zip(h, g)]
        rho = torch.full((len(h),), 1e-3)
        for i in dead:  # no step at the largest rho: inactive from the second iteration on
            ees[i][:] = float("nan")
            rho[i] = 10.0
        rho, ee = rho.cuda(), torch.cat(ees).cuda()
        st, it = (torch.zeros(k * len(h), dtype=torch.int32, device="cuda") for k in (1, 3))
        s = _solver(pkg, h)
        try:
            s.batch_sqp(xu, lam, ee, rho, 3, st, it)
            torch.cuda.synchronize()
            out.append([t.cpu().numpy() for t in (xu, lam, rho, st, it)])
        finally:
            s.close()
    n, T = len(horizons), sum(horizons)
    assert all(bool(out[0][3][i] & pkg.ST_ACTIVE) == (i not in dead) for i in range(n))
    for a, b, m in zip(*out, (21 * T - 7 * n, 14 * T, n, n, 3 * n)):
        assert np.array_equal(a[:m], b[:m], equal_nan=a.dtype.kind == "f")
    assert (out[0][4].reshape(n, 3)[[i for i in range(n) if i not in dead]] > 0).all()
