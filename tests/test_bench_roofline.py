"""bench.py's roofline of the timed region, on the CPU: the kernel that the timed
steps run (steps in registers), its recorded counters, and the canonical step's
bytes over the same time."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


@pytest.mark.parametrize("config,n,nb,nf", [("water1M", 3, 10**6, 0), ("hetero200k", 5, 200000, 500000)])
def test_timed_regions_kernel_has_records(config, n, nb, nf):
    r = bench.steps_roofline(0.02, n, nb, nf, config)
    valu, traffic = bench.recorded("valu", "steps", config), bench.recorded("traffic", "steps", config)
    assert valu["kernel"] == traffic["kernel"] == "k_steps" and valu["boundaries_per_launch"] == 64
    assert r["kernel"] == "steps"
    assert r["achieved"] == pytest.approx(valu["valu_instr_per_launch"] / 64 / 0.02e-3 / 1e9)
    assert r["frac"] == pytest.approx(r["achieved"] / bench.VALU_PEAK_G)
    assert r["frac_hbm"] == pytest.approx(traffic["bytes_per_launch"] / 64 / 0.02e-3 / 8e12)
    assert r["canonical_bytes_per_step"] == nb * (128 + 36 * n) + nf * 64 + 36 * (n * nb + nf)


def test_without_records():
    r = bench.steps_roofline(0.1, 3, 4 * 10**6, 0, "water4M")
    assert r["frac"] is None and r["frac_hbm"] is None and r["canonical_frac_hbm"] > 0
