"""What bench.py divides its kernel times by: the algorithmic bytes of a step's
passes, and the share of the timed steps that store every field."""
import os
import sys

import pytest

from weldformgpu_amd import _abi

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_inner_steps_count_what_they_move():
    inner, kept = bench.alg_bytes(False, False, 0.0), bench.alg_bytes(False, False, 1.0)
    # x v m rho h -> rho; -> 9 rates; x v sigma rho Cs h -> a; x v a u ID -> x v u
    assert (inner["dens"], inner["rates"], inner["accel"], inner["integrate"]) == (80, 144, 144, 172)
    # the rates are neither read back nor stored, the acceleration is neither
    assert inner["rates_stress"] == inner["rates"] + inner["stress"] - 2 * 72 - 8  # rho once
    assert inner["accel_integrate"] == inner["accel"] + inner["integrate"] - 2 * 24 - 48
    # p, sigma_eq, the strain rate and sigma; a; drho, dT/dt, T_b
    assert kept["stress"] - inner["stress"] == 72
    assert kept["rates_stress"] - inner["rates_stress"] == 72 + 72
    assert kept["accel_integrate"] - inner["accel_integrate"] == 24
    assert kept["cond_dens"] - inner["cond_dens"] == 24
    mixed = bench.alg_bytes(True, False, 0.0)
    assert all(mixed[k] < inner[k] for k in ("dens", "rates", "stress", "accel", "cond_dens"))
    assert bench.alg_bytes(True, True, 0.0)["rates"] == mixed["rates"] + 24  # the normals


@pytest.mark.parametrize("contact,stale,policy,first,steps,kept", [
    (0, True, 0, 3000, 20, [19]),
    (0, False, 0, 3000, 20, [4, 9, 14, 19]),
    (1, True, 0, 3000, 20, [0, 4, 5, 9, 10, 14, 15, 19]),
    (1, False, 0, 3002, 6, [2, 3, 5]),
    (1, True, 1, 3000, 20, list(range(20))),
])
def test_share_of_steps_that_store_every_field(contact, stale, policy, first, steps, kept):
    cfg = _abi.default_config()
    cfg.contact, cfg.rebuild_policy = contact, policy
    if not stale:
        cfg.quirks &= ~_abi.WF_Q_STALE_NS_POS
    assert bench.kept_share(cfg, first, steps) == len(kept) / steps
