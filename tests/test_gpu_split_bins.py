"""GPU: the split-form PCG's packing.  Few instances are spread over the
device (a bin each), many share bins of up to eight; either way an instance
is solved bitwise the same."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _solve(pkg, horizons, max_items, seed, tol=1e-5):
    n, T = len(horizons), int(sum(horizons))
    s = pkg.Solver(pkg.default_config(max_knots=max(horizons), max_instances=n, max_total_knots=T, pcg_exit_tol=tol))
    try:
        s.batch_setup(horizons)
        s.batch_set_plan(max_items=max_items)
        g = torch.Generator().manual_seed(seed)
        L = 21 * T - 7 * n
        xu = (0.3 * torch.randn(L, generator=g)).cuda()
        lam = (0.01 * torch.randn(14 * T, generator=g)).cuda()
        ee = torch.rand(6 * T, generator=g).cuda()
        rho = torch.full((n,), 1e-3, device="cuda")
        st = torch.zeros(n, dtype=torch.int32, device="cuda")
        it = torch.zeros(2 * n, dtype=torch.int32, device="cuda")
        s.batch_sqp(xu, lam, ee, rho, 2, st, it)
        torch.cuda.synchronize()
        return s.batch_pcg_layout()["bins"], [t.cpu().numpy() for t in (xu, lam, rho, st, it)]
    finally:
        s.close()


def test_shared_bins_are_bitwise_single_bins(pkg):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    # more instances than a device has compute units, so bins are shared:
    # horizons at the edges of a group (8 knots), a wave (32) and the longest
    horizons = ([2, 3, 7, 8, 9, 15, 16, 17, 31, 32] * 150 + [33, 63, 64, 65, 127, 128, 129, 255, 256])
    bins8, a = _solve(pkg, horizons, 8, 3)
    bins1, b = _solve(pkg, horizons, 1, 3)
    assert bins1 == len(horizons) and bins8 < bins1 / 4
    for x, y in zip(a, b):
        assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f")
    assert (a[4] > 0).any()


def test_few_instances_get_a_bin_each(pkg):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    horizons = [64] * 40 + [5, 97, 256]
    bins, a = _solve(pkg, horizons, 8, 4)
    assert bins == len(horizons)
    # the same instances inside a batch that shares bins
    many = horizons + [2] * 4000
    bins_many, b = _solve(pkg, many, 8, 4)
    assert bins_many < len(many) / 4
    # inputs are drawn per layout, so only the layout's own repeat is compared
    _, c = _solve(pkg, many, 1, 4)
    for x, y in zip(b, c):
        assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f")
