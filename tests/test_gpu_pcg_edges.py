"""GPU: the on-chip PCG kernels of a single instance (one workgroup for N <=
128, with 1, 2 or 4 knots per lane row; teams of two and four workgroups above)
at the edges of their layouts, from a non-zero start, against the fp64 oracle.

A fixed number of iterations (the exit test cannot be met), so both sides
take the same steps.  Bound: 4 x the distance of the oracle's fp32 twin, or
1e-5 where that is less: six iterations of sums of at most 42 terms and of 14 N
products keep to some 1e-6 in fp32, while a row, block or neighbour taken
wrongly shows at 1e-2 and above."""
import numpy as np
import pytest

import helpers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 133, 255, 256, 257, 511, 512])
def test_fixed_iterations(solver, orc, N):
    x0, ee, xu = helpers.make_instance(orc, 700 + N, N)
    cfg = orc.make_cfg()
    G, Cm, g, c = orc.form_kkt(cfg, N, xu.astype(np.float64), ee.astype(np.float64), xu[:14].astype(np.float64))
    S, P, gam, _ = (np.asarray(a, np.float32) for a in orc.form_schur(N, G, Cm, g, c, 1e-3))
    lam0 = (0.01 * np.random.default_rng(N).standard_normal(14 * N)).astype(np.float32)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (S, P, gam, lam0)]
    it = torch.zeros(1, dtype=torch.int32, device="cuda")
    fl = torch.zeros(1, dtype=torch.int32, device="cuda")
    solver.pcg(N, dev[0], dev[1], dev[2], dev[3], 6, 0.0, it, fl)
    got = dev[3].cpu().numpy().astype(np.float64)
    want, it_o, _ = orc.pcg(N, S, P, gam, lam0.astype(np.float64), 6, 0.0)
    twin, _, _ = orc.pcg(N, S, P, gam, lam0, 6, 0.0, dtype=np.float32)
    err, floor = helpers.rel_err(got, want), helpers.rel_err(twin, want)
    print(f"N={N} rel(gpu, oracle)={err:.2e} twin={floor:.2e}")
    assert int(it.item()) == it_o == 6 and int(fl.item()) == 1
    assert err < max(1e-5, 4 * floor)
