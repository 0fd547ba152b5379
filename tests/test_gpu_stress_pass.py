"""The rates pass that updates its particles' stress as soon as their sums are
done, and what a call's inner steps leave unstored.

The fused pass takes domains with one h, with the Newton return map those of
64 particles a workgroup at least and 768 tiles at most.  Tolerances: three
steps against the FP64 oracle, relative L2 <= 1e-9 (FP64: rounding of ~56
terms a sum, grown by the steps' differences of neighbouring values) and 1e-4
(mixed: FP32 terms).
"""
import numpy as np
import pytest

from weldformgpu_amd import _abi, scenarios
from weldformgpu_amd.domain import WfError

from harness import MECH_FIELDS, randomize, rel_l2, to_gpu, to_oracle

pytestmark = pytest.mark.gpu

TOL = {_abi.WF_FP64: 1e-9, _abi.WF_MIXED: 1e-4}


def _scenario(n, precision, newton, beta=0.0):
    """The first n particles of a thermo-mechanical cylinder at yield."""
    sc = scenarios.c3_johnson_cook(scale=0.3 if n < 20000 else 0.51)
    for k, v in sc.fields.items():
        sc.fields[k] = v[:n].copy()
    sc.cfg.n_particles = sc.cfg.solid_count = n
    sc.cfg.precision = precision
    sc.cfg.return_map = _abi.WF_RETURN_NEWTON if newton else _abi.WF_RETURN_REFERENCE
    randomize(sc, seed=n, v_scale=0.5)
    sc.fields["T"] = 300.0 + np.random.default_rng(n).uniform(0.0, 50.0, n)
    return sc


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("newton", [True, False])
@pytest.mark.parametrize("n", [1, 129, 4097, 8192, 8193, 16384, 16385, 98304, 98305])
def test_stress_update_in_the_rates_pass(oracle, wflib, n, newton, precision):
    sc = _scenario(n, precision, newton)
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    st.step(sc.cfg, sc.bcs, 3)
    fused = not newton or 8192 < n <= 98304
    with to_gpu(sc, wflib) as d:
        d.set_timing(True)
        d.step(3)
        assert d.kernel_time("rates_stress")[1] == (3 if fused else 0)
        assert d.kernel_time("stress")[1] == (0 if fused else 3)
        for k in MECH_FIELDS:
            if np.linalg.norm(st[k]) > 0.0:
                assert rel_l2(d.get(k), st[k]) <= TOL[precision], k


FIELDS = MECH_FIELDS + ["T"]


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("contact", [False, True])
def test_one_call_leaves_what_single_steps_leave(wflib, contact, precision):
    """A call's inner steps store less; every field at its end is that of as
    many single-step calls, bit for bit."""
    runs = []
    for calls in ([7], [1] * 7):
        if contact:
            sc = scenarios.c4_contact(scale=0.2, r=0.25e-3, dens=16, offset=0.137)
            sc.cfg.precision = precision
            randomize(sc, seed=3, v_scale=0.5)
        else:
            sc = _scenario(9000, precision, True)
        with to_gpu(sc, wflib) as d:
            for k in calls:
                d.step(k)
            runs.append({k: d.get(k) for k in FIELDS})
    for k in FIELDS:
        assert np.array_equal(runs[0][k], runs[1][k]), k


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
def test_call_that_a_rebuild_ends(wflib, precision):
    """A particle flies off, and the rebuild at the sixth step refuses the
    domain: the fields are those of the five steps before it."""
    def case():
        sc = _scenario(3000, precision, False)
        sc.cfg.quirks &= ~_abi.WF_Q_STALE_NS_POS
        sc.cfg.ns_min_plastic = 0.0
        sc.fields["pl_strain"] = np.full(sc.n, 1e-3)
        sc.fields["v"][np.flatnonzero(sc.fields["ID"] == 0)[-1]] = [0.0, 0.0, 1e13]
        return sc
    runs = []
    with to_gpu(case(), wflib) as d:
        d.nsearch()
        with pytest.raises(WfError):
            d.step(20)
        assert d.stats()["step"] == 5
        runs.append({k: d.get(k) for k in FIELDS})
    with to_gpu(case(), wflib) as d:
        d.nsearch()
        for _ in range(5):
            d.step(1)
        runs.append({k: d.get(k) for k in FIELDS})
    for k in FIELDS:
        assert np.array_equal(runs[0][k], runs[1][k], equal_nan=True), k


@pytest.mark.parametrize("contact", [False, True])
@pytest.mark.parametrize("n", [3000, 9000, 17000])
def test_fp64_integration_in_the_acceleration_pass(wflib, n, contact):
    """FP64: each particle integrated in the acceleration pass (those with
    contact candidates in the contact pass) against the separate pass, over
    steps with rebuilds: the same arithmetic in the same order, so every field
    is bit-identical.  A domain with two masses keeps the separate pass."""
    runs = []
    for fuse, masses in ((1, 1), (0, 1), (1, 2)):
        if contact:
            scale = (n / 1320424) ** (1 / 3)
            sc = scenarios.c4_contact(scale=scale, dens=max(6, int(64 * scale)), offset=0.137)
            randomize(sc, seed=n, v_scale=0.5)
        else:
            sc = _scenario(n, _abi.WF_FP64, True)
        sc.cfg.precision = _abi.WF_FP64
        sc.cfg.fuse_integrate = fuse
        sc.cfg.quirks &= ~_abi.WF_Q_STALE_NS_POS
        sc.cfg.ns_min_plastic = 0.0
        sc.fields["pl_strain"] = np.full(sc.n, 1e-3)
        if masses == 2:
            sc.fields["m"] = sc.fields["m"] * np.where(np.arange(sc.n) == 5, 1.0 + 1e-6, 1.0)
        with to_gpu(sc, wflib) as d:
            d.set_timing(True)
            for k in (1, 7, 3):
                d.step(k)
            runs.append({k: d.get(k) for k in FIELDS + (["contforce"] if contact else [])})
            fused = fuse and masses == 1
            assert d.kernel_time("accel_integrate")[1] == (11 if fused else 0)
            assert d.kernel_time("integrate")[1] == (0 if fused else 11)
            assert d.stats()["ns_builds"] >= 2
            if contact:
                assert (d.get("cont_nb_count") > 0).sum() > 0
    for k in runs[0]:
        assert np.array_equal(runs[0][k], runs[1][k]), k
        if k != "a":  # a mass 1e-6 apart: the same physics by the other passes
            assert rel_l2(runs[2][k], runs[0][k]) < 1e-4, k


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("field", ["G", "rho0", "Cs", "m"])
def test_constants_that_differ(oracle, wflib, field, precision):
    """With one rest density, shear modulus, mass and sound speed the stress
    update reads none of the four planes; a particle apart brings them back."""
    sc = _scenario(9000, precision, True)
    uniform = sc.fields[field].copy()
    sc.fields[field][4321] *= 1.01
    st = to_oracle(oracle, sc)
    st.nsearch(sc.cfg)
    st.step(sc.cfg, sc.bcs, 2)
    apart = sc.fields[field].copy()
    sc.fields[field] = uniform
    with to_gpu(sc, wflib) as d:
        d.set(field, apart)
        d.step(2)
        for k in MECH_FIELDS:
            if np.linalg.norm(st[k]) > 0.0:
                assert rel_l2(d.get(k), st[k]) <= TOL[precision], k


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
def test_call_that_a_candidate_search_ends(wflib, precision):
    """The rigid mesh, far from the particles, turns non-finite in mid-call, and
    the candidate search of the sixth step refuses it (the lists, rebuilt from
    an unchanged snapshot, end no call).  The fields are those that single-step
    calls leave, which have the step's passes up to the acceleration, and the
    Newton statistics count the step."""
    def case(omega):
        sc = scenarios.c4_contact(scale=0.2, r=0.25e-3, dens=16, offset=0.137)
        sc.cfg.precision = precision
        randomize(sc, seed=4, v_scale=0.5)
        sc.fields["T"] = 300.0 + np.random.default_rng(4).uniform(0.0, 50.0, sc.n)
        sc.meshes[0]["nodes"][:, 2] += 1.0
        sc.meshes[0]["vel"] = (0.0, 0.0, 0.0)
        # the nodes' distance grows by a factor of omega dt a step
        sc.meshes[0]["omega"] = (0.0, 0.0, omega / sc.cfg.dt)
        return sc
    fields = FIELDS + ["Ta", "Tb", "dTdt", "contforce", "normal"]
    runs, newton = [], []
    for calls in ([20], [1] * 6):
        with to_gpu(case(1e65), wflib) as d:
            for k in calls[:-1]:
                d.step(k)
            with pytest.raises(WfError, match="non-finite rigid mesh"):
                d.step(calls[-1])
            assert d.stats()["step"] == 5
            newton.append(d.stats()["newton_calls"])
            runs.append({k: d.get(k) for k in fields})
    for k in fields:
        assert np.array_equal(runs[0][k], runs[1][k]), k
    with to_gpu(case(0.0), wflib) as d:
        d.step(5)
        before = d.get("a")
        d.step(1)
        assert newton == [d.stats()["newton_calls"]] * 2 and newton[0] > 0
        for k in ("sigma", "strrate", "rho", "pl_strain"):
            assert np.array_equal(runs[0][k], d.get(k)), k
    assert not np.array_equal(runs[0]["a"], before)  # of the step the search ended


@pytest.mark.parametrize("n", [3000, 9000, 17000])
def test_mixed_contact_integration_in_the_acceleration_pass(wflib, n):
    """Mixed precision: contact steps that integrate in the acceleration pass
    (the particles with contact candidates in the contact pass) against the
    separate pass, over steps with rebuilds: bit-identical, the positions that
    are updated in place and what the next steps read of the spare mirrors
    included."""
    runs = []
    for fuse in (1, 0):
        scale = (n / 1320424) ** (1 / 3)
        sc = scenarios.c4_contact(scale=scale, dens=max(6, int(64 * scale)), offset=0.137)
        randomize(sc, seed=n, v_scale=0.5)
        sc.cfg.precision = _abi.WF_MIXED
        sc.cfg.fuse_integrate = fuse
        sc.cfg.quirks &= ~_abi.WF_Q_STALE_NS_POS
        sc.cfg.ns_min_plastic = 0.0
        sc.fields["pl_strain"] = np.full(sc.n, 1e-3)
        with to_gpu(sc, wflib) as d:
            d.set_timing(True)
            for k in (1, 7, 3):
                d.step(k)
            runs.append({k: d.get(k) for k in FIELDS + ["contforce", "q_friction"]})
            assert d.kernel_time("accel_integrate")[1] == (11 if fuse else 0)
            assert d.kernel_time("integrate")[1] == (0 if fuse else 11)
            assert d.stats()["ns_builds"] >= 2
            assert (d.get("cont_nb_count") > 0).sum() > 0
            assert np.abs(runs[-1]["contforce"]).sum() > 0
    for k in runs[0]:
        assert np.array_equal(runs[0][k], runs[1][k]), k


@pytest.mark.parametrize("precision", [_abi.WF_FP64, _abi.WF_MIXED])
@pytest.mark.parametrize("field", ["G", "rho0", "Cs", "m", "h"])
@pytest.mark.parametrize("n,odd", [(65535, 65534), (65536, 0), (65536, 65535), (70001, 70000)])
def test_one_value_apart_in_large_domains(oracle, wflib, n, odd, field, precision):
    """From 65,536 values on the device finds out whether a field has one
    value: a particle apart at either end, and uniform values again after it."""
    sc = _scenario(n, precision, False)
    uniform = sc.fields[field].copy()
    st = to_oracle(oracle, sc)
    apart = uniform.copy()
    apart[odd] *= 1.01 if field != "h" else 1.0 + 1e-4
    st[field] = apart
    st.nsearch(sc.cfg)
    st.step(sc.cfg, sc.bcs, 1)
    with to_gpu(sc, wflib) as d:
        d.set(field, apart)
        d.step(1)
        for k in MECH_FIELDS:
            if np.linalg.norm(st[k]) > 0.0:
                assert rel_l2(d.get(k), st[k]) <= TOL[precision], k
        near = np.argsort(((sc.fields["x"] - sc.fields["x"][odd]) ** 2).sum(1))[:30]
        for k in ("v", "sigma", "rho"):  # where the particle apart shows
            assert rel_l2(d.get(k)[near], st[k][near]) <= TOL[precision], k
    runs = []
    for values in ([uniform], [apart, uniform]):
        with to_gpu(sc, wflib) as d:
            for v in values:
                d.set(field, v)
            d.step(2)
            runs.append({k: d.get(k) for k in FIELDS})
    for k in FIELDS:
        assert np.array_equal(runs[0][k], runs[1][k]), k
