"""Pair loops with the neighbours staged whole in LDS.

They take domains whose particles share one h, and in the acceleration one
sound speed (FP64: and one mass); other domains keep the gathering loops and
the general record.  Both must give the same passes at every tile remainder,
and a domain that changes from one to the other must not use stale records.
Up to 32, 64 and 128 tiles (4,096, 8,192 and 16,384 particles) a tile is dealt
out to 8, 4 and 2 workgroups.

Tolerances: against the FP64 oracle, one call, relative L2 <= 1e-12 (FP64:
rounding of ~56 terms a sum) and 2e-5 (mixed: FP32 terms).
"""
import numpy as np
import pytest

from weldformgpu_amd import _abi, scenarios

from harness import randomize, rel_l2, to_gpu, to_oracle

pytestmark = pytest.mark.gpu

TOL = {_abi.WF_FP64: 1e-12, _abi.WF_MIXED: 2e-5}


def _scenario(n, precision, beta):
    """The first n particles of a thermo-mechanical cylinder, random v, stress
    and temperature."""
    sc = scenarios.c3_johnson_cook(scale=0.3)
    for k, v in sc.fields.items():
        sc.fields[k] = v[:n].copy()
    sc.cfg.n_particles = sc.cfg.solid_count = n
    sc.cfg.precision = precision
    sc.cfg.beta = beta
    randomize(sc, seed=n)
    rng = np.random.default_rng(n)
    sc.fields["T"] = 300.0 + rng.uniform(0.0, 50.0, n)
    sc.fields["k_T"] = rng.choice([150.0, 200.0], n)
    return sc


def _large(n, precision):
    sc = scenarios.c3_johnson_cook(scale=0.46)
    for k, v in sc.fields.items():
        sc.fields[k] = v[:n].copy()
    sc.cfg.n_particles = sc.cfg.solid_count = n
    sc.cfg.precision = precision
    randomize(sc, seed=n)
    rng = np.random.default_rng(n)
    sc.fields["T"] = 300.0 + rng.uniform(0.0, 50.0, n)
    sc.fields["k_T"] = rng.choice([150.0, 200.0], n)
    return sc


def _passes(d, st, cfg, tol):
    d.CalcDensInc()
    st.calc_dens_inc(cfg)
    d.CalcRateTensors()
    st.calc_rate_tensors(cfg)
    d.CalcAccel()
    st.calc_accel(cfg)
    d.CalcTempInc()
    st.calc_temp_inc(cfg)
    for k in ("drho", "strrate", "rotrate", "a", "dTdt"):
        assert rel_l2(d.get(k), st[k]) <= tol, k


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("n", [1, 63, 127, 128, 129, 1000, 4096, 4097, 8192, 8193, 16384, 16385])
def test_uniform_and_general_passes(oracle, wflib, n, precision):
    sc = _scenario(n, precision, 1.0 if n == 129 else 0.0)
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    with to_gpu(sc, wflib) as d:
        d.nsearch()
        _passes(d, st, sc.cfg, TOL[precision])
        # one particle apart in Cs, then in m, then in h: the general loops
        for k, f in (("Cs", 1.01), ("m", 1.01), ("h", 1.0 + 1e-6)):
            a = st[k].copy()
            a[n // 2] *= f
            st[k] = a
            d.set(k, a)
            _passes(d, st, sc.cfg, TOL[precision])
        # and back
        for k in ("h", "m", "Cs"):
            st[k] = sc.fields[k]
            d.set(k, sc.fields[k])
        _passes(d, st, sc.cfg, TOL[precision])


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("n", [2000, 6000, 12000])
def test_large_sets_in_split_tiles(oracle, wflib, n, precision):
    """Staged sets left uncompacted, above the LDS set: the loops take them in
    passes, with 16, 8 and 4 lanes a particle."""
    sc = _scenario(n, precision, 0.0)
    sc.cfg.ns_compact_max = 256
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    with to_gpu(sc, wflib) as d:
        d.nsearch()
        _passes(d, st, sc.cfg, TOL[precision])


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("uniform_mass", [True, False])
def test_surface_sums_in_the_rates_pass(oracle, wflib, uniform_mass, precision):
    """A contact step takes the free-surface sums along in the rates pass when
    the masses are one, in a pass of its own when they are not."""
    sc = scenarios.c4_contact(scale=0.15, r=0.25e-3, dens=12, offset=0.137)
    sc.cfg.precision = precision
    randomize(sc, seed=5, v_scale=0.1, shear=False)
    if not uniform_mass:
        sc.fields["m"][sc.n // 3] *= 1.0 + 1e-9
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    st.step(sc.cfg, sc.bcs, 2)
    with to_gpu(sc, wflib) as d:
        d.step(2)
        assert np.array_equal(d.get("ID"), st["ID"])
        assert (d.get("ID") == sc.cfg.id_free_surf).sum() > 100
        assert rel_l2(d.get("normal"), st.contact_arrays["normal"]) <= TOL[precision]


@pytest.mark.parametrize("policy", [_abi.WF_REBUILD_EVERY_N, _abi.WF_REBUILD_PLASTIC_ZONE])
@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
def test_contact_pass_over_the_listed_particles(oracle, wflib, precision, policy):
    """Only particles with candidates take the contact pass: what a caller
    left in the others' contact force and friction heat is gone after a step,
    also when a reorder between two candidate searches moved the particles."""
    sc = scenarios.c4_contact(scale=0.2, r=0.25e-3, dens=16, offset=0.137)
    sc.cfg.precision = precision
    sc.cfg.fric_heat = 1.0
    sc.cfg.rebuild_policy = policy
    if policy != _abi.WF_REBUILD_EVERY_N:
        sc.cfg.ns_skin = 0.4 * sc.meta["dx"]
    sc.meshes[0]["nodes"][:, 2] -= 0.05 * sc.meta["dx"]
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    st.step(sc.cfg, sc.bcs, 7)
    with to_gpu(sc, wflib) as d:
        d.set("contforce", np.ones((sc.n, 3)))
        d.set("q_friction", np.full(sc.n, 1e3))
        d.step(2)
        d.snapshot_positions()
        d.nsearch()  # a reorder, two steps into the candidates' five
        cnt, cf = d.get("cont_nb_count"), d.get("contforce")
        assert 0 < (cnt > 0).sum() < sc.n
        assert not cf[cnt == 0].any() and not d.get("q_friction")[cnt == 0].any()
        d.step(5)
        tol = 1e-9 if precision == _abi.WF_FP64 else 1e-4
        cf = d.get("contforce")
        assert np.abs(cf).sum() > 0
        assert rel_l2(cf, st.contact_arrays["cf"]) <= tol
        for k in ("u", "v", "sigma"):
            assert rel_l2(d.get(k), st[k]) <= tol, k


@pytest.mark.parametrize("uniform_mass", [True, False])
def test_contact_timing_counts_what_was_launched(wflib, uniform_mass):
    """The contact timer's intervals: forces and mesh motion in every step, the
    candidate search in every fifth, and the free-surface pass where the rates
    pass does not take its sums along (in the search's interval)."""
    sc = scenarios.c4_contact(scale=0.2, r=0.25e-3, dens=16, offset=0.137)
    if not uniform_mass:
        sc.fields["m"][sc.n // 3] *= 1.0 + 1e-9
    with to_gpu(sc, wflib) as d:
        d.set_timing(True)
        d.step(10)
        assert d.kernel_time("contact")[1] == (2 * 10 + 2 if uniform_mass else 3 * 10)


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("n", [17000, 65536, 65537])
@pytest.mark.parametrize("compact_max", [1, 0])
def test_large_sets_of_whole_tiles(oracle, wflib, n, compact_max, precision):
    """Two lanes a particle, up to 512 tiles (65,536 particles) with 1,024 and
    beyond with 960 staged entries: sets left uncompacted (~1,230 particles),
    and, off the lattice under a list skin, sets on both sides of the two."""
    sc = _large(n, precision)
    if compact_max:
        sc.cfg.ns_compact_max = compact_max
    else:
        dx = sc.meta["dx"]
        sc.cfg.rebuild_policy = _abi.WF_REBUILD_PLASTIC_ZONE
        sc.cfg.ns_skin, sc.cfg.ep_hot = 0.3 * dx, 1e9
        sc.fields["x"] += np.random.default_rng(n).uniform(-0.2 * dx, 0.2 * dx, (n, 3))
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    with to_gpu(sc, wflib) as d:
        d.nsearch()
        assert d.nsearch_stats()[1] == 0
        _passes(d, st, sc.cfg, TOL[precision])
