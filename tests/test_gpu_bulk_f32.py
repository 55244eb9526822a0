"""Bulk updates in binary32 against the binary64 oracle: grids of one phase with
a rough mu, where every tile of the tile paths is bulk (k_bulk, from the tile's
flag and one phase's tables) and every cell of the one-hot path takes the light
mu sweep.

The tolerance.  With u = 2^-24 and m = max |mu|, loading rounds mu by at most
u m, which the diffusion step (lambda <= 1/4, a contraction) does not enlarge.
Each step reads five values of mu that lack their low parts, u m off each: four
face differences, hence 8 lambda u m, where lambda is the largest row sum of
dMu/dc D dc/dmu dt/dx^2; forming the increment and adding it rounds by at most
2 u m more (|increment| <= m)."""
import numpy as np
import pytest

import gputil
from eshwar_dipan_amd import gpstep

U = 2.0 ** -24


def _lambda(p, a):
    C = p.ncomp
    A = np.array([[p.A[a][i][j] * (2.0 if i == j else 1.0) for j in range(C)] for i in range(C)])
    D = np.array([[p.diffusivity[a][i][j] for j in range(C)] for i in range(C)])
    cmu = np.array([[p.cmu[a][i][j] for j in range(C)] for i in range(C)])
    return float(np.abs(A @ D @ cmu).sum(axis=1).max()) * p.dt / min(p.dx, p.dy) ** 2


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["path 0", "path 3", "path 6", "ensemble"])
@pytest.mark.parametrize("P,C", [(2, 1), (3, 2), (4, 1)])
def test_gpu_bulk_f32_matches_oracle(P, C, where):
    steps = 9
    print(f"\n[gpu] bulk grids in binary32, P={P} C={C}, {where}", flush=True)
    inps = [gputil.make_params(P=P, C=C, mesh=(67 + 30 * a, 131), bc=(1, 1, 3, 3), extra=("DELTA_X = 0.8;",) * (a % 2),
                               gabc=0.5 if P > 2 else None, D_sol=0.4) for a in range(P)]
    states = []
    for a, inp in enumerate(inps):
        p = inp.p
        phi = np.zeros((P, p.mesh_x, p.mesh_y))
        phi[a] = 1.0
        states.append((phi, 0.8 + 0.05 * np.random.default_rng(a).standard_normal((C, p.mesh_x, p.mesh_y))))
    if where == "ensemble":
        e = gpstep.Ensemble(inps, "f32")
        for a in range(P):
            e.set_state(a, *states[a])
        e.step(steps)
        out = [e.get_state(a) for a in range(P)]
        assert e.sched_info()[1] == 0
        e.close()
    else:
        out = []
        for a in range(P):
            s = gpstep.Solver(inps[a], "f32", path=int(where[-1]))
            s.set_state(*states[a])
            s.step(steps)
            out.append(s.get_state())
            if where != "path 6":
                assert s.sched_info()[1] == 0
            s.close()
    for a in range(P):
        phi, mu = gputil.oracle_run(inps[a].p, *states[a], steps)
        lam, m = _lambda(inps[a].p, a), float(np.abs(states[a][1]).max())
        tol = U * m * (1 + steps * (8 * lam + 2))
        err, moved = float(np.abs(out[a][1] - mu).max()), float(np.abs(mu - states[a][1]).max())
        print(f"  phase {a}: lambda {lam:.3f}, error {err:.2e} of {tol:.2e}, mu moved by {moved:.2e}", flush=True)
        assert lam <= 0.25 and np.array_equal(out[a][0], phi)
        assert err <= tol
