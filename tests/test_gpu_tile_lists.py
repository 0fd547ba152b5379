"""The list builder's two ways to a tile's cells (flags over the box around
them, a sort where the box is too large) and its candidate filter, against the
oracle's lists: bit-exact."""
import numpy as np
import pytest

from weldformgpu_amd import scenarios

from harness import to_gpu, to_oracle

pytestmark = pytest.mark.gpu


def _cloud(n, cells, seed):
    """n random particles in a cube of about `cells` search cells an edge."""
    sc = scenarios.c3_johnson_cook(scale=0.3)
    for k, v in sc.fields.items():
        sc.fields[k] = v[:n].copy()
    sc.cfg.n_particles = sc.cfg.solid_count = n
    rng = np.random.default_rng(seed)
    sc.fields["x"] = rng.uniform(0.0, cells * 2.02 * sc.cfg.h_glob, (n, 3))
    # coincident particles are no neighbours of each other
    sc.fields["x"][n // 2] = sc.fields["x"][0]
    return sc


# cells an edge: dense tiles of a few cells, tiles over most of the domain, and
# tiles whose box holds more than 4,096 cells
@pytest.mark.parametrize("cells", [1.5, 6.0, 15.0, 40.0, 300.0])
@pytest.mark.parametrize("n", [2, 63, 129, 700, 5000])
def test_lists_of_random_clouds(oracle, wflib, n, cells):
    if n / cells**3 > 12.0:
        n = int(12 * cells**3)  # below the list cap
    sc = _cloud(n, cells, seed=n)
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    oc, _, ol = st.neighbor_rows()
    with to_gpu(sc, wflib) as d:
        d.nsearch()
        gc, _, gl = d.neighbors()
        assert np.array_equal(gc, oc) and np.array_equal(gl, ol)
