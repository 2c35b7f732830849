"""The benchmark's operation counts: the route and the arithmetic that the energy ran on decide both."""
import pytest

import bench


@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16x3", "int8"])
def test_energy_work_follows_the_route(form):
    W, M, N, K = 7, 20, 5, 90
    NM = N * M
    # over the table: every entry of half the square and K traces, a multiply-add of a complex G each
    assert bench.energy_work(form, True, W, M, N, K) == (W * 4 * (NM * NM / 2 + NM * K), 78.6)
    flop, peak = bench.energy_work(form, False, W, M, N, K)
    real_products = {"fp64": 2, "fp32": 4, "bf16x3": 9, "int8": 2}[form]   # of a multiply-add of T_n
    assert flop == W * K * N * N * M * 2 * real_products
    assert peak == {"fp64": 78.6, "fp32": 157.3, "bf16x3": 2500.0, "int8": None}[form]


def test_energy_roofline_weighs_each_call_by_its_own_peak():
    rate, frac = bench.energy_roofline([(2e9, 100.0, 0.05), (9e9, 1000.0, 0.15)])
    assert rate == pytest.approx(11e9 / 0.2 / 1e9)
    assert frac == pytest.approx((0.02 + 0.009) / 0.2)      # ms at the peaks over the ms taken
    assert bench.energy_roofline([(2e9, 100.0, 0.05), (9e9, None, 0.15)]) == (pytest.approx(55.0), None)
    assert bench.energy_roofline([]) == (0.0, None)


def test_gate_sees_the_contractions_that_the_forms_change():
    dE = {"fp32": 0.0, "bf16x3": 0.0, "int8": 2e-10}     # over the pair table E_loc is FP64's
    errors = {"fp32": {"vbias": 1.1e-6, "vHS": 1.5e-6}, "bf16x3": {"vbias": 8.0e-6, "vHS": 7.9e-6},
              "int8": {"vbias": 1.1e-6, "vHS": 4.1e-6}}
    assert bench.meets_gate("fp64", {}, {})
    assert bench.meets_gate("fp32", dE, errors)
    assert not bench.meets_gate("bf16x3", dE, errors)
    assert not bench.meets_gate("int8", dE, errors)
    assert not bench.meets_gate("fp32", {"fp32": 1e-5}, errors)
    assert not bench.meets_gate("fp32", dE, {}) and not bench.meets_gate("fp32", {}, errors)
