"""GPU: split-form PCG of short instances, spread over twice the SIMDs (all
N <= 64, no more instances than compute units or few waves), against the bins of
eight knots per row, which an instance of N = 65 in the batch selects: bitwise
the same, from a non-zero lambda, at the edges of a group (8 knots), of a wave
(16) and of the range."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

HORIZONS = [2, 3, 4, 5, 6, 7, 8, 9, 10, 15, 16, 17, 24, 25, 31, 32, 33, 47, 48, 49, 56, 57, 63, 64]


def _solve(pkg, horizons, tol, max_iter):
    n, T = len(horizons), int(sum(horizons))
    s = pkg.Solver(pkg.default_config(max_knots=max(horizons), max_instances=n, max_total_knots=T, pcg_exit_tol=tol,
                                      pcg_max_iter=max_iter))
    try:
        s.batch_setup(horizons)
        g = [torch.Generator().manual_seed(100 + N) for N in horizons]
        xu = torch.cat([0.3 * torch.randn(21 * N - 7, generator=q) for N, q in zip(horizons, g)]).cuda()
        lam = torch.cat([0.01 * torch.randn(14 * N, generator=q) for N, q in zip(horizons, g)]).cuda()
        ee = torch.cat([torch.rand(6 * N, generator=q) for N, q in zip(horizons, g)]).cuda()
        rho = torch.full((n,), 1e-3, device="cuda")
        st = torch.zeros(n, dtype=torch.int32, device="cuda")
        it = torch.zeros(2 * n, dtype=torch.int32, device="cuda")
        s.batch_sqp(xu, lam, ee, rho, 2, st, it)
        torch.cuda.synchronize()
        return [t.cpu().numpy() for t in (xu, lam, rho, st, it)]
    finally:
        s.close()


@pytest.mark.parametrize("horizons", [HORIZONS, [16] * 150 + [3] * 350], ids=["a unit each", "many"])
@pytest.mark.parametrize("tol,max_iter", [(1e-5, 1000), (0.0, 7), (0.0, 1)])
def test_short_kernel_is_bitwise_the_bins(pkg, tol, max_iter, horizons):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    T, n = sum(horizons), len(horizons)
    a = _solve(pkg, horizons, tol, max_iter)
    b = _solve(pkg, horizons + [65], tol, max_iter)
    for x, y, m in zip(a, b, (21 * T - 7 * n, 14 * T, n, n, 2 * n)):
        assert np.array_equal(x[:m], y[:m], equal_nan=x.dtype.kind == "f")
    assert (a[4] > 0).any()
