"""The wing solve's product with the inverse at the edges of its workgroups: 64 rows each, 16 wavefronts
over the columns.  Bar of the wing tests: 1e-11 on circulations and force."""
import numpy as np
import pytest

from uvlm_amd.vlm import Wing, reference_wing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129])
def test_solve(orc, n):
    from oracle import vlm
    V, U = reference_wing(npanels=n), np.array([0.0, 1.0, 0.0])
    print(f"[wing] n={n}", flush=True)
    w, ow = Wing(V), vlm.Wing(V)
    assert ow.n == n
    g, F = w.solve(None, U)
    eg = vlm.solve(ow, U, np.zeros((n, 3)))
    eF = vlm.force(ow, eg, U, np.zeros((n, 3)))
    assert np.linalg.norm(g - eg) < 1e-11 * np.linalg.norm(eg) and np.linalg.norm(F - eF) < 1e-11 * np.linalg.norm(eF)
