"""GPU: direct-mode batches with refined Schur solves (direct_refine = 2) and a
refined KKT step, which solves again on the factors that the first solve left:
eliminated from both ends up to two instances of the longest horizon per compute
unit in all, from one end above.  Ragged, from N = 2, with an inactive instance, against the fp64 oracle's
direct SQP step, and on both sides of the line against single solves."""
import numpy as np
import pytest

import helpers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture
def make_solver(pkg):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    made = []

    def make(horizons):
        s = pkg.Solver(pkg.default_config(max_knots=max(horizons), max_instances=len(horizons),
                                          max_total_knots=sum(horizons), flags=pkg.FLAG_DIRECT_SOLVE, direct_refine=2,
                                          direct_kkt_refine=1, sqp_max_iter=2))
        made.append(s)
        return s

    yield make
    for s in made:
        s.close()


def _batch(s, horizons, xus, ees, rhos):
    n, T = len(horizons), sum(horizons)
    xu, lam = torch.from_numpy(np.concatenate(xus)).cuda(), torch.zeros(14 * T, device="cuda")
    rho, st = torch.tensor(rhos, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    s.batch_setup(horizons)
    s.batch_sqp(xu, lam, torch.from_numpy(np.concatenate(ees)).cuda(), rho, 2, st)
    torch.cuda.synchronize()
    kx, kl = np.cumsum([0] + [21 * N - 7 for N in horizons]), np.cumsum([0] + [14 * N for N in horizons])
    xu, lam = xu.cpu().numpy(), lam.cpu().numpy()
    return ([xu[a:b] for a, b in zip(kx, kx[1:])], [lam[a:b] for a, b in zip(kl, kl[1:])], st.cpu().numpy())


def test_ragged_batch_vs_oracle(make_solver, pkg, orc):
    horizons, dead = [64, 2, 17, 3, 130, 4, 33, 256, 5], 6
    inst = [helpers.make_instance(orc, 4100 + i, N) for i, N in enumerate(horizons)]
    xus, ees = [i[2] for i in inst], [i[1] for i in inst]
    bad = [e.copy() for e in ees]
    bad[dead][:] = np.nan
    rhos = [1e-3] * len(horizons)
    rhos[dead] = 10.0  # at the largest: no step in the first iteration ends it, so it is inactive in the second
    s = make_solver(horizons)
    xu, _, st = _batch(s, horizons, xus, bad, rhos)
    assert not st[dead] & pkg.ST_ACTIVE
    assert np.array_equal(xu[dead], xus[dead])
    for i, N in enumerate(horizons):
        if i == dead:
            continue
        ref = orc.sqp_solve(orc.make_cfg(sqp_max_iter=2), N, ees[i].astype(np.float64), np.zeros(14 * N),
                            xus[i].astype(np.float64), 1e-3, use_direct=True)
        err = helpers.rel_err(xu[i], ref["xu"])
        print(f"N={N} rel(xu)={err:.2e}")
        assert err < 1e-4, N  # as the plain direct SQP (test_gpu_direct.py): exact to fp32 storage, measured ~1e-6


@pytest.mark.parametrize("per_unit", [2, 4])
def test_both_sides_of_the_line_match_single_solves(make_solver, pkg, orc, per_unit):
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    kinds = [2, 3, 4, 13, 16, 15, 16]
    horizons = [kinds[(3 * i) % len(kinds)] for i in range(per_unit * n_cu)]
    assert (sum(horizons) > 2 * n_cu * max(horizons)) == (per_unit == 4)
    inst = {N: helpers.make_instance(orc, 4200 + N, N) for N in kinds}
    s = make_solver(horizons)
    xu, lam, st = _batch(s, horizons, [inst[N][2] for N in horizons], [inst[N][1] for N in horizons],
                         [1e-3] * len(horizons))
    for N, (_, ee, xu0) in inst.items():
        x, l = torch.from_numpy(xu0).cuda(), torch.zeros(14 * N, device="cuda")
        s.sqp_solve(N, torch.from_numpy(ee).cuda(), l, x, 1e-3)
        torch.cuda.synchronize()
        x, l = x.cpu().numpy(), l.cpu().numpy()
        same = [i for i, h in enumerate(horizons) if h == N]
        for i in same:
            assert np.array_equal(xu[i], xu[same[0]]) and np.array_equal(lam[i], lam[same[0]])
        # refined steps: to fp32 storage (the bound of the batched direct test)
        assert helpers.rel_err(xu[same[0]], x) < 1e-5 and helpers.rel_err(lam[same[0]], l) < 1e-5, N
