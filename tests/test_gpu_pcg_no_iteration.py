"""GPU: a PCG that takes no iteration (a cap of 0, or a start that already
meets the tolerance) leaves lambda as it was, also entries that are not finite:
one-workgroup kernel, resident kernel (stair), teams of two and four."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stair", [False, True])
@pytest.mark.parametrize("N", [2, 32, 64, 128, 200, 300])
def test_lambda_is_untouched(pkg, N, stair):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    s = pkg.Solver(pkg.default_config(max_knots=N, max_total_knots=N, flags=pkg.FLAG_PCG_STAIR if stair else 0))
    try:
        S = torch.zeros(N, 3, 14, 14)
        S[:, 1] = -2.0 * torch.eye(14)
        P = torch.zeros(N, 3, 14, 14)
        P[:, 1] = -0.5 * torch.eye(14)
        g = torch.Generator().manual_seed(N)
        lam = torch.randn(14 * N, generator=g)
        gamma = -2.0 * lam  # S lambda = gamma already
        S, P, gamma = S.reshape(-1).cuda(), P.reshape(-1).cuda(), gamma.cuda()
        it, fl = (torch.full((1,), 9, dtype=torch.int32, device="cuda") for _ in range(2))
        for cap, bad in ((5, ()), (0, ()), (0, (float("inf"), float("-inf"))), (0, (float("nan"),))):
            x = lam.clone()
            for k, v in enumerate(bad):
                x[(5 + 9 * k) % (14 * N)] = v
            d = x.cuda()
            s.pcg(N, S, P, gamma, d, cap, 1e-5 if cap else 0.0, it, fl)
            torch.cuda.synchronize()
            assert np.array_equal(d.cpu().numpy(), x.numpy(), equal_nan=True), (cap, bad)
            assert int(it) == 0 and int(fl) == (0 if cap else 1)
    finally:
        s.close()
