"""The window kernels (one fine k3 per lane, J windows in LDS) against the CPU oracle, the plain
FP64 form bit for bit and the FMA-FP64 form at its bar, and the FP32-compensated form against the
sweep kernel bit for bit, where they can go wrong: every count of
source multipoles L, rows below m, fields with fewer L than the other, T or E alone, odd l
counts against the groups of 8 and 4, k3 counts that leave partial tiles, one step over several
windows, J rows with an index_xmin_J of their own, and a batch whose k3 lie too far apart.
"""
import numpy as np
import pytest

from song_amd import lib as L
from tests.conftest import field_errors, run_oracle

BASE = dict(has_T=1, has_E=1, m_list=[0, 1, 2], l_max_los_t=4, l_max_los_p=4, k_size=3,
            k_min=2e-3, k_max=0.01, k3_size=9, tau_size=37, l_size=9, l_max=140, dk_fine=2.5e-5,
            xx_max=200.0)
CASES = {
    "L_0_T": dict(BASE, has_E=0, m_list=[0], l_max_los_t=0),
    "L_1": dict(BASE, l_max_los_t=1, l_max_los_p=1, m_list=[0, 1]),
    "L_2": dict(BASE, l_max_los_t=2, l_max_los_p=2),
    "L_3_m_0_3": dict(BASE, l_max_los_t=3, l_max_los_p=3, m_list=[0, 3]),
    "L_4_5": dict(BASE, l_max_los_p=5, l_size=5),
    "L_6_4": dict(BASE, l_max_los_t=6, l_size=13),
    "L_7_m_0_to_5": dict(BASE, l_max_los_t=7, l_max_los_p=7, m_list=[0, 1, 2, 3, 4, 5]),
    "E_without_B": dict(BASE, has_T=0, m_list=[0], l_size=17),
    "m_above_L": dict(BASE, l_max_los_t=2, l_max_los_p=2, m_list=[1, 4], l_size=6),
    "linear_flat_3_l": dict(BASE, k3_interpolation=L.LINEAR, extrapolation=L.FLAT_EXTRAP,
                            extra_osc_left=2.0, extra_osc_right=2.0, l_size=3),
    "wide_steps": dict(BASE, k_max=0.02, dk_fine=1.2e-4, xx_max=400.0),
    "one_tile": dict(BASE, k_size=2, k_min=0.004, k_max=0.008, k3_size=12, dk_fine=1e-2),
}


def _run(cfg, oracle, overrides=()):
    def scenario():
        s = L.Scenario(cfg)
        for o in overrides:
            s.override_J(*o)
        return s

    ref = run_oracle(scenario(), oracle)
    s = scenario()
    s.prepare()
    eng = L.Engine(0)
    eng.load(s)
    ran = []
    for kt in (64, 32, 16):
        print(f"tile of {kt}", flush=True)
        try:
            eng.set_shape(L.FORM_FP64, 3, kt, 8, 0)
        except L.LosError:
            continue
        eng.run()
        eng.store(s)
        assert np.array_equal(s.gather(), ref), f"tile of {kt}"
        ran.append(kt)
    eng.set_form(L.FORM_FP64_FAST)
    tt2 = ref.size // int(s.k3_sizes()[:, 0].sum())
    for kt in ran:  # the same sums with FMA, at the form's bar
        eng.set_shape(L.FORM_FP64_FAST, 3, kt, 8, 0)
        eng.run()
        eng.store(s)
        assert field_errors(s.gather(), ref, tt2).max() < 1e-12, f"FMA, tile of {kt}"
    eng.close()
    s.close()
    return ref, ran


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_window_equals_oracle(name, oracle):
    print(f"case {name}", flush=True)
    ref, ran = _run(L.Config(**CASES[name]), oracle)
    assert 16 in ran
    if name in ("L_6_4", "L_7_m_0_to_5"):
        assert ran == [64, 32, 16]
    if name != "m_above_L":
        assert np.count_nonzero(ref) > 0.1 * ref.size


def _same_as_sweep(cfg, overrides=()):
    s = L.Scenario(cfg)
    for o in overrides:
        s.override_J(*o)
    s.prepare()
    eng = L.Engine(0)
    eng.set_form(L.FORM_FP32C)
    eng.load(s)
    eng.set_shape(L.FORM_FP32C, 1, 2, 1, 0)
    eng.run()
    eng.store(s)
    ref, ran = s.gather(), []
    for kt in (64, 32, 16):
        print(f"tile of {kt}", flush=True)
        try:
            eng.set_shape(L.FORM_FP32C, 3, kt, 8, 0)
        except L.LosError:
            continue
        eng.run()
        eng.store(s)
        assert np.array_equal(s.gather(), ref), f"tile of {kt}"
        ran.append(kt)
    eng.close()
    s.close()
    assert 16 in ran


@pytest.mark.gpu
@pytest.mark.parametrize("tau_size", [31, 32, 33, 70])
@pytest.mark.parametrize("name", list(CASES))
def test_fp32_window_equals_sweep(name, tau_size):
    """Counts of time steps about the 32 of a partial sum."""
    print(f"case {name} {tau_size} steps", flush=True)
    _same_as_sweep(L.Config(**dict(CASES[name], tau_size=tau_size)))


@pytest.mark.gpu
def test_window_rows_with_their_own_first_point(oracle):
    """J rows of one l whose first stored points are far apart: the skip holds row by row."""
    cfg = L.Config(**dict(BASE, l_size=6))
    s = L.Scenario(cfg)
    rng = np.random.default_rng(3)
    n_x = int(cfg.xx_max / cfg.xx_step + 1)
    over = []
    for jt in range(3):
        for Lv in range(cfg.l_max_los_t + 1):
            xmin = int(rng.integers(1, 300))
            over.append((jt, Lv, 2, 0, xmin, rng.normal(size=n_x - xmin)))
    s.close()
    _, ran = _run(cfg, oracle, over)
    assert 16 in ran
    _same_as_sweep(cfg, over)


@pytest.mark.gpu
def test_window_not_offered_to_sparse_k3():
    """k3 hundreds of x points apart: the shape is refused with a message, the tuner runs."""
    cfg = L.Config(**dict(BASE, k_max=0.1, dk_fine=2e-2, k3_size=4, xx_max=1500.0))
    s = L.Scenario(cfg)
    s.prepare()
    eng = L.Engine(0)
    eng.load(s)
    with pytest.raises(L.LosError):
        eng.set_shape(L.FORM_FP64, 3, 64, 8, 0)
    eng.run()
    assert eng.get_shape(L.FORM_FP64)[0] != 3
    eng.close()
    s.close()
