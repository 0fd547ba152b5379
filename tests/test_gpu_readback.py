"""Fields of 12 MiB and more come back through pinned chunks by several host
threads: every value, at sizes round the threshold and the 1 MiB chunk."""
import numpy as np
import pytest

from weldformgpu_amd import _abi
from weldformgpu_amd.domain import Domain

pytestmark = pytest.mark.gpu


# n x 6 doubles: one below 12 MiB, 12 MiB, one chunk and a bit more, many
@pytest.mark.parametrize("n", [262143, 262144, 284000, 1000003])
def test_large_fields_come_back_whole(wflib, n):
    cfg = _abi.default_config()
    cfg.n_particles = cfg.solid_count = n
    cfg.h_glob = cfg.dt = 1.0
    rng = np.random.default_rng(n)
    with Domain(cfg, wflib) as d:
        for k, c in (("sigma", 6), ("v", 3), ("T", 1)):
            a = rng.standard_normal((n, c) if c > 1 else n)
            d.set(k, a)
            for _ in range(2):
                assert np.array_equal(d.get(k), a), k


# the ends of a chunk's 16-byte words: 4, 8 and 12 bytes over, and a last chunk
# shorter than a word
@pytest.mark.parametrize("n", [262145, 349526, 3145729, 3145731])
def test_last_words_come_back(wflib, n):
    cfg = _abi.default_config()
    cfg.n_particles = cfg.solid_count = n
    cfg.h_glob = cfg.dt = 1.0
    rng = np.random.default_rng(n)
    with Domain(cfg, wflib) as d:
        for k, a in (("sigma", rng.standard_normal((n, 6))), ("rho", rng.standard_normal(n)),
                     ("ID", rng.integers(-2**31, 2**31 - 1, n, dtype=np.int32))):
            d.set(k, a)
            out = d.get(k)
            assert np.array_equal(out, a), k
