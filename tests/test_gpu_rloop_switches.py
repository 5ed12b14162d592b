"""The radial loop under combinations of its switches that no dump of the
reference holds, and at the shortest and longest rows of its grid stage's slot
form (n_phi = 24: one lane per slot and 32 theta rows per block, the last
block partly filled; n_phi = 1536: 64 lanes per slot), against the oracle's
radial loop.  Bar: 1e-11, that of the loop's other comparisons with the oracle
(the Lorentz force and Coriolis terms cancel a few digits)."""
import numpy as np
import pytest

from conftest import rel_l2
from magic_amd import sht, workload
import rloop_cases as rc

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _case(case, L, **switches):
    ph = dict(rc.phys_of(rc.load(case)), **switches)
    nlev = 2
    fields = {n: None for n in sht.RLOOP_IN}
    fields.update(dict(zip(sht.NL_INPUTS, workload.nl_inputs(L, nlev, stream=13))))
    fields["xi"] = np.stack([workload.coefficients(L, 13, 20, i, potential=False) for i in range(nlev)])
    fields["phi"] = np.stack([workload.coefficients(L, 13, 21, i, potential=False) for i in range(nlev)])
    r = np.array([0.8, 1.2])
    one = np.ones(nlev)
    rad = {"r": r, "or1": 1 / r, "or2": 1 / r ** 2, "or4": 1 / r ** 4, "orho1": 1 / (1 + 0.1 * r),
           "beta": -0.1 / (1 + 0.1 * r), "otemp1": 1 / (1.5 - 0.2 * r), "visc": one, "lambda": 1 + 0.1 * r,
           "temp0": one, "epscProf": one, "delxr2": np.full(nlev, 1e-3), "delxh2": np.full(nlev, 2e-2),
           "nR": np.array([5, 9], dtype=np.int32), "l_R": np.array([L, L - 2], dtype=np.int32)}
    return ph, rad, fields


def _run(ph, rad, fields, L, nt, nph):
    p = sht.Plan(L, nt, nph, max_levels=2)
    outs = {n: np.zeros((2, p.lm_max), dtype=np.complex128) for n in rc.outputs_of(ph)}
    dtr, dth = np.zeros(2), np.zeros(2)
    sht.rloop(p, ph, 2, rad, fields, outs, dtr, dth)
    p.close()
    return outs, dtr, dth


def _compare(got, ph, rad, fields, L, nt, nph):
    from oracle import oracle
    from rloop_reference import oracle_rloop
    want, wtr, wth = oracle_rloop(oracle.Plan(L, nt, nph), ph, 2, rad, fields, 1)
    outs, dtr, dth = got
    assert set(outs) == set(want)
    for n in outs:
        assert rel_l2(outs[n], want[n]) < TOL, n
    assert rel_l2(dtr, wtr) < TOL and rel_l2(dth, wth) < TOL


PHASE = dict(l_phase_field=1, epsPhase=0.03, penaltyFac=0.5, tmelt=0.11)
SWITCHES = {
    "outside_the_conductor": ("bouss_mhd", dict(n_r_LCR=6)),
    "outside_the_conductor_anelastic": ("anel_mhd", dict(n_r_LCR=6)),
    "lorentz_force_alone": ("bouss_mhd", dict(l_conv_nl=0)),
    "lorentz_force_alone_phase": ("bouss_mhd", dict(PHASE, l_conv_nl=0)),
    "lorentz_force_alone_outside": ("bouss_mhd", dict(PHASE, l_conv_nl=0, n_r_LCR=6)),
    "curl_viscous_heating": ("anel_mhd", dict(l_adv_curl=1)),
    "linear_heat": ("bouss_mhd", dict(l_heat_nl=0)),
    "composition_without_curl": ("doublediff", dict(l_adv_curl=0)),
    "phase_without_curl": ("phase", dict(l_adv_curl=0)),
}


@pytest.mark.parametrize("L,nt,nph", [(15, 24, 48), (20, 36, 160), (20, 36, 768)])
@pytest.mark.parametrize("name", SWITCHES)
def test_switch_combinations_match_oracle(name, L, nt, nph):
    base, switches = SWITCHES[name]
    print("switches", name, L, nt, nph, flush=True)
    ph, rad, fields = _case(base, L, **switches)
    _compare(_run(ph, rad, fields, L, nt, nph), ph, rad, fields, L, nt, nph)


@pytest.mark.parametrize("case,L,nt,nph", [(c, 7, 36, 24) for c in rc.CASES] +
                         [(c, 12, 20, 1536) for c in ("doublediff", "precession", "phase")])
def test_slot_ends_match_oracle(case, L, nt, nph):
    print("ends", case, L, nt, nph, flush=True)
    ph, rad, fields = _case(case, L)
    _compare(_run(ph, rad, fields, L, nt, nph), ph, rad, fields, L, nt, nph)


@pytest.mark.parametrize("L,nt,nph", [(15, 24, 48), (20, 36, 160)])
def test_linear_heat_ignores_the_entropy(L, nt, nph):
    """Without nonlinear heat advection u s is not formed: an entropy that is not
    finite leaves no trace in the outputs."""
    ph, rad, fields = _case("bouss_mhd", L, l_heat_nl=0)
    bad = dict(fields, s=fields["s"].copy())
    bad["s"][1, 3] = np.inf
    got = _run(ph, rad, bad, L, nt, nph)
    assert np.all(got[0]["dVSrLM"] == 0.0)
    _compare(got, ph, rad, fields, L, nt, nph)
