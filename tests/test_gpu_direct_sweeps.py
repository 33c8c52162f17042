"""GPU: the wave-per-instance direct solve at the edges of its sweeps (the
factorisation alternates two buffers by knot, the substitution takes four
knots a turn and three turns ahead), with pivots whose inverse is taken by
division, and with a workspace at an odd multiple of four bytes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _system(N, seed):
    """-S block tridiagonal, symmetric, diagonally dominant: condition below 10."""
    rng = np.random.default_rng(seed)
    diag = np.zeros((N, 14, 14), np.float32)
    left = np.zeros((N, 14, 14), np.float32)
    for b in range(N):
        m = rng.uniform(-0.05, 0.05, (14, 14))
        diag[b] = (-(2.0 * np.eye(14) + m + m.T)).astype(np.float32)
        diag[b] = (diag[b] + diag[b].T) / 2
        if b:
            left[b] = rng.uniform(-0.03, 0.03, (14, 14)).astype(np.float32)
    S = np.zeros((N, 3, 14, 14), np.float32)  # blocks transposed below: column-major
    S[:, 1] = diag.transpose(0, 2, 1)
    S[1:, 0] = left[1:].transpose(0, 2, 1)
    S[:-1, 2] = left[1:]
    full = np.zeros((14 * N, 14 * N))
    for b in range(N):
        full[14 * b:14 * b + 14, 14 * b:14 * b + 14] = diag[b]
        if b:
            full[14 * b:14 * b + 14, 14 * b - 14:14 * b] = left[b]
            full[14 * b - 14:14 * b, 14 * b:14 * b + 14] = left[b].T
    gamma = rng.uniform(-1, 1, 14 * N).astype(np.float32)
    return S.reshape(-1), gamma, np.linalg.solve(full, gamma.astype(np.float64))


def _solve(pkg, N, S, gamma, refine, offset=0):
    s = pkg.Solver(pkg.default_config(max_knots=max(N, 2), max_total_knots=max(N, 2)))
    try:
        lam = torch.empty(14 * N, device="cuda")
        work = torch.empty(588 * N + 4, device="cuda")[offset:offset + 588 * N]
        s.direct_solve(N, torch.from_numpy(S).cuda(), torch.from_numpy(gamma).cuda(), lam, refine, work)
        torch.cuda.synchronize()
        return lam.cpu().numpy()
    finally:
        s.close()


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 15, 16, 17, 24, 25, 37])
def test_sweep_edges(pkg, N):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    S, gamma, ref = _system(N, N)
    for offset in (0, 1):
        # condition below 10: two refinements leave the rounding of lambda and
        # of its last sum, 2 x 2^-24 relative to the largest entry
        lam = _solve(pkg, N, S, gamma, 2, offset)
        assert np.abs(lam - ref).max() <= 1.3e-7 * np.abs(ref).max() + 1e-9, (N, offset)
    # without refinement: a 14 N deep chain of fp32 sums at condition below 10
    lam = _solve(pkg, N, S, gamma, 0)
    assert np.abs(lam - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("exponent", [-60, 60])
def test_pivots_outside_the_quick_range(pkg, exponent):
    """S and gamma scaled by a power of two give the same lambda, bitwise; at
    2^-60 and 2^60 every pivot's inverse comes from the division instead."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N = 13
    S, gamma, _ = _system(N, 99)
    scale = np.float32(2.0 ** exponent)
    for refine in (0, 2):
        a = _solve(pkg, N, S, gamma, refine)
        b = _solve(pkg, N, S * scale, gamma * scale, refine)
        assert np.array_equal(a, b), (exponent, refine)
