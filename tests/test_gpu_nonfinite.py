"""A value that is not finite reaches the particles that list its owner and no
others.

A lane takes its particle's list by quads, and what fills a quad past the
list's end must not bring in another particle's values: 0 x NaN is NaN.  The
domains are clusters of ten particles, all within reach of each other (lists of
nine) and out of reach of the next cluster, so a tile holds about thirteen
clusters, and whatever one of them holds must leave the others bit-identical.
At 3,000, 6,000, 12,000 and 19,000 particles a tile is dealt out to 8, 4, 2
workgroups and 1.
"""
import numpy as np
import pytest

from weldformgpu_amd import _abi, scenarios

from harness import to_gpu

pytestmark = pytest.mark.gpu

PER = 10  # particles a cluster


def _clusters(n, precision, seed):
    sc = scenarios.c3_johnson_cook(scale=0.3)
    for k, v in sc.fields.items():
        sc.fields[k] = v[:n].copy()
    sc.cfg.n_particles = sc.cfg.solid_count = n
    sc.cfg.precision = precision
    h = sc.cfg.h_glob
    rng = np.random.default_rng(seed)
    nc = n // PER
    edge = int(np.ceil(nc ** (1 / 3)))
    at = np.stack(np.unravel_index(np.arange(nc), (edge,) * 3), 1) * (8.0 * h)
    d = rng.standard_normal((n, 3))
    d *= (0.9 * h * rng.uniform(0.3, 1.0, n) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]
    sc.fields["x"] = np.repeat(at, PER, 0) + d
    sc.fields["v"] = rng.uniform(-0.1, 0.1, (n, 3))
    ss = rng.uniform(-1e7, 1e7, (n, 6))
    ss[:, 2] = -(ss[:, 0] + ss[:, 1])
    sc.fields["shearstress"] = ss
    sc.fields["sigma"] = ss.copy()
    sc.fields["T"] = 300.0 + rng.uniform(0.0, 50.0, n)
    sc.fields["k_T"] = rng.choice([150.0, 200.0], n)
    bad = rng.choice(nc, max(1, nc // 4), replace=False) * PER + rng.integers(0, PER, max(1, nc // 4))
    hit = np.zeros(n, bool)
    hit[(bad[:, None] // PER * PER + np.arange(PER)).ravel()] = True
    return sc, bad, hit


# what each value must reach: the outputs that are NaN in every neighbour
REACHES = {"v": ("drho", "strrate", "rotrate"), "sigma": ("a",), "T": ("dTdt",), "x": ()}
OUT = ("drho", "strrate", "rotrate", "a", "dTdt")


def _passes(d):
    d.CalcDensInc()
    d.CalcRateTensors()
    d.CalcAccel()
    d.CalcTempInc()
    return {k: d.get(k) for k in OUT}


def _check_passes(wflib, n, precision, apart):
    sc, bad, hit = _clusters(n, precision, seed=n)
    for k, f in apart.items():
        sc.fields[k][n // 3] *= f
    with to_gpu(sc, wflib) as d:
        d.nsearch()
        cnt, _, _ = d.neighbors()
        assert (cnt == PER - 1).all()
        clean = _passes(d)
        for k, reached in REACHES.items():
            for value in (np.nan, np.inf):
                a = sc.fields[k].copy()
                a[bad] = value
                d.set(k, a)
                got = _passes(d)
                for o in OUT:
                    assert np.isfinite(got[o][~hit]).all(), (k, value, o)
                    # (in mixed precision a tile's frame is its first particle's
                    # cell: without one the others round in another frame)
                    if k != "x" or precision == _abi.WF_FP64:
                        assert np.array_equal(got[o][~hit], clean[o][~hit]), (k, value, o)
                    if o in reached and np.isnan(value):
                        nb = hit.copy()
                        nb[bad] = False
                        assert np.isnan(got[o][nb]).reshape(nb.sum(), -1).any(1).all(), (k, o)
            d.set(k, sc.fields[k])


def _check_steps(wflib, n, precision, apart):
    sc, bad, hit = _clusters(n, precision, seed=n + 1)
    for k, f in apart.items():
        sc.fields[k][n // 3] *= f
    runs = []
    for k in (None, "v", "T", "shearstress"):
        with to_gpu(sc, wflib) as d:
            if k:
                a = sc.fields[k].copy()
                a[bad] = np.nan
                d.set(k, a)
            d.step(3)
            runs.append({o: d.get(o) for o in ("x", "v", "a", "rho", "sigma", "pl_strain", "T")})
        for o, a in runs[-1].items():
            assert np.isfinite(a[~hit]).all(), (k, o)
            assert np.array_equal(a[~hit], runs[0][o][~hit]), (k, o)


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("n", [60, 3000, 6000, 12000, 19000])
def test_passes_with_one_h(wflib, n, precision):
    _check_passes(wflib, n, precision, {})


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("n", [60, 3000, 6000, 12000, 19000])
def test_steps_with_one_h(wflib, n, precision):
    _check_steps(wflib, n, precision, {})


# the loops that gather: one particle's h, sound speed or mass apart
@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("apart", ["h", "Cs", "m"])
@pytest.mark.parametrize("n", [60, 6000, 19000])
def test_passes_of_general_domains(wflib, n, apart, precision):
    _check_passes(wflib, n, precision, {apart: 1.0 + 1e-6})


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("apart", ["h", "Cs", "m"])
@pytest.mark.parametrize("n", [60, 6000, 19000])
def test_steps_of_general_domains(wflib, n, apart, precision):
    _check_steps(wflib, n, precision, {apart: 1.0 + 1e-6})
