"""GPU: the receding-horizon shift of the closed loop at the edges of its
chunks (384 lanes of 16 elements: N = 293 is the last horizon whose plan fits
one), against the plan of the same SQP shifted on the host.  Whole numbers of
elements move, so the comparison is exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_traj", [True, False])
@pytest.mark.parametrize("N", [2, 3, 64, 293, 294, 440, 512])
def test_one_step_shifts_the_plan(pkg, N, with_traj):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    s = pkg.Solver(pkg.default_config(max_knots=512, max_instances=1, max_total_knots=512))
    try:
        x0, ee, traj = s.track_inputs(90 + N, 1, N)
        xu, lam = traj[:21 * N - 7].clone(), torch.zeros(14 * N, device="cuda")
        s.batch_setup([N])
        rho = torch.full((1,), s.cfg.rho_reset, device="cuda")
        st = torch.zeros(1, dtype=torch.int32, device="cuda")
        plan, plan_lam = xu.clone(), lam.clone()
        plan[:14] = x0
        s.batch_sqp(plan, plan_lam, ee[:6 * N].clone(), rho, 1, st)
        plan, plan_lam = plan.cpu().numpy(), plan_lam.cpu().numpy()
        cl = pkg.default_closed_loop(steps=1, sqp_iters=1, noise_sigma=1e-3, substeps=3)
        states, err, _, _ = s.closed_loop(N, x0, ee, xu, lam, cl, traj if with_traj else None)
        torch.cuda.synchronize()
    finally:
        s.close()
    states, traj = states.cpu().numpy(), traj.cpu().numpy()
    want = plan.copy()
    want[:-21] = plan[21:]
    tail = slice(21 * (N - 2) + 14, 21 * N - 7)
    want[tail] = traj[21 * (N - 1) + 14:21 * N + 14] if with_traj else np.concatenate([np.zeros(7), plan[-14:]])
    want[:14] = states[1]
    want_lam = np.concatenate([plan_lam[14:], plan_lam[-14:]])
    assert np.array_equal(xu.cpu().numpy(), want)
    assert np.array_equal(lam.cpu().numpy(), want_lam)
    assert np.isfinite(err.cpu().numpy()).all()
