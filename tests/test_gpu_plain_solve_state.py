"""GPU: what a plain solve leaves in the handle that the batch calls read."""
import numpy as np
import pytest

import helpers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _batch_sqp(pkg, orc, s, horizons, seed, iters):
    inst = [helpers.make_instance(orc, seed + i, N) for i, N in enumerate(horizons)]
    s.batch_setup(horizons)
    xu, ee = _dev(np.concatenate([i[2] for i in inst])), _dev(np.concatenate([i[1] for i in inst]))
    lam, rho = torch.zeros(14 * sum(horizons), device="cuda"), torch.full((len(horizons),), 1e-3, device="cuda")
    st, it = (torch.zeros(k * len(horizons), dtype=torch.int32, device="cuda") for k in (1, iters))
    s.batch_sqp(xu, lam, ee, rho, iters, st, it)
    return it


def _pcg_exit(s, n):
    it, fl = (torch.full((n,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    eta = torch.full((n,), -1.0, device="cuda")
    s.batch_pcg_exit(it, fl, eta)
    torch.cuda.synchronize()
    return it.cpu().numpy(), fl.cpu().numpy(), eta.cpu().numpy()


@pytest.mark.parametrize("graph", [False, True])
def test_exit_state_is_the_last_solves(pkg, orc, graph):
    """mpc_batch_pcg_exit: iterations, flag and eta of one and the same solve,
    a plain one's for instance 0 if that was the last."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    s = pkg.Solver(pkg.default_config(max_knots=64, max_instances=2, max_total_knots=128, pcg_max_iter=150,
                                      sqp_max_iter=2))
    try:
        s.batch_set_graph(graph)
        horizons, K = [64, 32], 2
        first = _batch_sqp(pkg, orc, s, horizons, 5500, K)
        before = _pcg_exit(s, 2)
        assert np.array_equal(before[0], first.cpu().numpy().reshape(2, K)[:, -1])
        _, ee, xu = helpers.make_instance(orc, 5600, 16)
        s.set_config(pcg_max_iter=7, pcg_exit_tol=0.0)
        iters = s.sqp_solve(16, _dev(ee), torch.zeros(14 * 16, device="cuda"), _dev(xu), 1e-3)[0]
        after = _pcg_exit(s, 2)
        assert after[0][0] == iters[1] == 7 and after[1][0] == 1
        assert after[0][1] == before[0][1] and after[1][1] == before[1][1] and after[2][1] == before[2][1]
        again = _pcg_exit(s, 2)
        assert all(np.array_equal(a, b) for a, b in zip(after, again))
        s.set_config(pcg_max_iter=150, pcg_exit_tol=1e-5)
        _batch_sqp(pkg, orc, s, horizons, 5500, K)
        last = _pcg_exit(s, 2)
        assert all(np.array_equal(a, b) for a, b in zip(before, last))
    finally:
        s.close()


@pytest.mark.parametrize("split", [0, 1])
def test_failed_plain_solve_leaves_the_batch_systems(pkg, orc, split):
    """A plain solve that ends at its first merit (a reference that is not
    finite) has solved nothing: the last batch's systems are still there."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    horizons = [64, 32]
    s = pkg.Solver(pkg.default_config(max_knots=64, max_instances=2, max_total_knots=128, sqp_max_iter=2))
    try:
        s.batch_set_plan(split=split)
        _, ee, xu = helpers.make_instance(orc, 5700, 64)
        s.sqp_solve(64, _dev(ee), torch.zeros(14 * 64, device="cuda"), _dev(xu), 1e-3)
        _batch_sqp(pkg, orc, s, horizons, 5800, 2)
        lam = [torch.zeros(14 * sum(horizons), device="cuda") for _ in range(3)]
        s.batch_direct_resolve(lam[0], refine=2)
        bad = torch.full((6 * 64,), float("nan"), device="cuda")
        for k in (1, 2):
            with pytest.raises(pkg.MpcError):
                s.sqp_solve(64, bad, torch.zeros(14 * 64, device="cuda"), _dev(xu), 1e-3)
            s.batch_direct_resolve(lam[k], refine=2)
        torch.cuda.synchronize()
        assert torch.isfinite(lam[0]).all() and lam[0].any()
        assert torch.equal(lam[0], lam[1]) and torch.equal(lam[0], lam[2])
    finally:
        s.close()
