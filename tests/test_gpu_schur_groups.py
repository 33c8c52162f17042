"""GPU: Schur formation at the edges of its workgroups (15 block rows each, the
inverses handed on from the group before) against the oracle, with the bounds
of test_form_schur: fp32 products of 14 terms and one 14 x 14 inverse against
fp64."""
import numpy as np
import pytest

import helpers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [14, 15, 16, 17, 29, 30, 31, 45, 46, 47])
def test_form_schur_workgroup_edges(solver, orc, N):
    x0, ee, xu = helpers.make_instance(orc, 800 + N, N)
    cfg = orc.make_cfg()
    G, Cm, g, c = orc.form_kkt(cfg, N, xu.astype(np.float64), ee.astype(np.float64), xu[:14].astype(np.float64))
    S, P, gam, Gi = orc.form_schur(N, *(np.asarray(a, np.float32).astype(np.float64) for a in (G, Cm, g, c)), 1e-3)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.float32))).cuda()
    dG, dS, dP = dev(G), torch.full((588 * N,), 7.0, device="cuda"), torch.full((588 * N,), 7.0, device="cuda")
    dg = torch.zeros(14 * N, device="cuda")
    solver.form_schur(N, dG, dev(Cm), dev(g), dev(c), dS, dP, dg, 1e-3)
    host = lambda t: t.cpu().numpy().astype(np.float64)
    for got, want in ((dS, S), (dP, P), (dg, gam), (dG, Gi)):
        got, want = host(got), np.asarray(want, np.float64)
        n = min(len(got), len(want))
        assert helpers.rel_err(got[:n], want[:n]) < 5e-4
    # block by block: a block taken from the wrong row shows at 1 in its own row
    for got, want in ((dS, S), (dP, P)):
        a, b = host(got).reshape(N, -1), np.asarray(want, np.float64).reshape(N, -1)
        assert (np.linalg.norm(a - b, axis=1) <= 1e-2 * np.linalg.norm(b, axis=1) + 1e-6).all()
