"""Response fields of many orbits reach the host in batches; each orbit's are those of the orbit alone."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


# fewer cells than a workgroup turns, as many, several workgroups; more orbits than one 64 MB batch holds at
# 16^2 (6553), the last of a batch and the first of the next among those compared
@pytest.mark.parametrize("level,n", [(3, 70), (4, 6600), (5, 3)])
@pytest.mark.parametrize("precision", [32, 64])
def test_fields_of_every_batch(level, n, precision):
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=0.05, level=level)
    w = model.make_workload(cfg, n=500, target_samples=20000)
    print(f"[gpu] fields out level={level} n={n} precision={precision}", flush=True)
    g = GalicGPU(w)
    i = np.arange(n) % w.n
    args = lambda i: (w.pos[i], w.vel[i], w.mass[i], w.tint[i], w.ptype[i])
    f = g.orbit_responses(*args(i), precision=precision)["fields"]
    again = g.orbit_responses(*args(i[:3]), precision=precision)["fields"]
    for k in np.unique(np.clip([0, 1, 2, n // 2, 6552, 6553, n - 1], 0, n - 1)):
        j = i[k:k + 1]
        one = g.orbit_responses(*args(j), precision=precision)["fields"]
        np.testing.assert_array_equal(f[k], one[0])
        if k < 3:
            np.testing.assert_array_equal(again[k], one[0])
    g.close()
