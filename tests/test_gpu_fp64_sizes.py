"""The FP64 transforms and nonlinear step at the edges of their kernels'
tiles against the FP64 oracle: every row-FFT length class (64 P points by
waves, slots of 1 to 64 lanes, generic passes), theta counts that leave the
last tile or row group partly empty, truncations whose l tiles need one or
several workgroups, level counts around the groups of 8, cut-offs below
l_max.  Bar: 1e-12 relative L2 per output, the FP64 form's throughout."""
import numpy as np
import pytest

from conftest import rel_l2
from magic_amd import sht, workload
from nl_reference import oracle_step, radial
import rloop_cases as rc

pytestmark = pytest.mark.gpu

TOL = 1e-12

# (l_max, n_theta, n_phi, minc): n_phi = 64 P for P = 1, 2, 3, 4, 5, 6, 8, 9, 10,
# 12, 15, 16, 18, 20, 24, then other lengths, then one and two groups of degrees
# in the analysis
GRIDS = [(13, 20, 64, 1), (20, 36, 128, 1), (42, 64, 128, 1), (31, 52, 192, 1), (85, 128, 256, 1),
         (20, 68, 320, 1), (33, 84, 384, 2), (30, 60, 512, 1), (20, 44, 576, 1), (21, 36, 640, 1),
         (20, 100, 768, 4), (11, 20, 960, 1), (20, 32, 1024, 1), (12, 20, 1152, 1), (15, 28, 1280, 1),
         (10, 20, 1536, 1), (15, 24, 48, 1), (31, 48, 96, 1), (26, 40, 80, 1), (33, 100, 400, 1),
         (282, 424, 64, 16), (283, 428, 64, 16), (345, 520, 64, 16)]


@pytest.mark.parametrize("L,nt,nph,minc", GRIDS)
def test_levels_batched_match_oracle(L, nt, nph, minc):
    """torpol_to_spat and spat_to_qst over 9 levels (one past a group of 8),
    two of them cut below l_max; scalar and per-level calls of one level."""
    import torch
    from oracle import oracle
    nlev = 9
    print("grid", L, nt, nph, minc, flush=True)
    p = sht.Plan(L, nt, nph, minc=minc, max_levels=nlev)
    o = oracle.Plan(L, nt, nph, minc=minc)
    lcut = [L] * nlev
    lcut[3], lcut[8] = L // 2, L - 1
    co = [np.stack([workload.coefficients(L, 5, f, i, minc=minc) for i in range(nlev)]) for f in range(3)]
    dev = torch.device("cuda")
    tin = [torch.from_numpy(x).to(dev) for x in co]
    g = [torch.zeros((nlev, nph, nt), dtype=torch.float64, device=dev) for _ in range(3)]
    p.torpol_to_spat_batch(*tin, lcut, *g)
    c = [torch.zeros_like(tin[0]) for _ in range(3)]
    p.spat_to_qst_batch(*g, lcut, *c)
    for i in range(nlev):
        want = o.torpol_to_spat(co[0][i], co[1][i], co[2][i], lcut[i])
        back = o.spat_to_qst(*want, lcut[i])
        for k in range(3):
            assert rel_l2(g[k][i].cpu().numpy(), want[k]) < TOL, (i, k)
            assert rel_l2(c[k][i].cpu().numpy(), back[k]) < TOL, (i, k)
    for a, b in ((p.scal_to_grad_spat(co[0][0], L), o.scal_to_grad_spat(co[0][0], L)),
                 (p.torpol_to_dphspat(co[0][1], co[1][1], L), o.torpol_to_dphspat(co[0][1], co[1][1], L)),
                 (p.spat_to_sphertor(want[1], want[2], L), o.spat_to_sphertor(want[1], want[2], L))):
        for k in range(2):
            assert rel_l2(a[k], b[k]) < TOL, k
    p.close()


@pytest.mark.parametrize("nlev", [128, 129])
def test_cutoffs_of_many_levels(nlev):
    """Every level's own cut-off at the number of levels whose cut-offs travel
    with the launch, and one past it."""
    import torch
    from oracle import oracle
    L, nt, nph = 10, 16, 64
    p = sht.Plan(L, nt, nph, max_levels=nlev)
    o = oracle.Plan(L, nt, nph)
    lcut = [1 + i % L for i in range(nlev)]
    co = [np.stack([workload.coefficients(L, 6, f, i) for i in range(nlev)]) for f in range(3)]
    dev = torch.device("cuda")
    tin = [torch.from_numpy(x).to(dev) for x in co]
    g = [torch.zeros((nlev, nph, nt), dtype=torch.float64, device=dev) for _ in range(3)]
    p.torpol_to_spat_batch(*tin, lcut, *g)
    c = [torch.zeros_like(tin[0]) for _ in range(3)]
    p.spat_to_qst_batch(*g, lcut, *c)
    for i in range(nlev):
        want = o.torpol_to_spat(co[0][i], co[1][i], co[2][i], lcut[i])
        back = o.spat_to_qst(*want, lcut[i])
        for k in range(3):
            assert rel_l2(g[k][i].cpu().numpy(), want[k]) < TOL, (i, k)
            assert rel_l2(c[k][i].cpu().numpy(), back[k]) < TOL, (i, k)
    p.close()


# the grid stage's forms: slots of 2, 4, 8, 16, 32, 64 lanes (two of them with
# several theta rows per workgroup, the last one partly filled), waves per
# component (n_phi = 256, 512, 1024), block-wide passes (128, 160)
@pytest.mark.parametrize("L,nt,nph,minc,nlev", [
    (15, 24, 48, 1, 3), (15, 28, 96, 1, 2), (42, 64, 128, 1, 3), (21, 36, 160, 1, 2), (64, 96, 192, 1, 2),
    (85, 128, 256, 1, 2), (30, 44, 384, 1, 2), (30, 52, 512, 1, 2), (64, 100, 768, 1, 2), (33, 60, 1024, 1, 2),
    (341, 512, 1024, 1, 1)])
def test_nl_step_matches_oracle(L, nt, nph, minc, nlev):
    import torch
    from oracle import oracle
    print("step", L, nt, nph, minc, nlev, flush=True)
    p = sht.Plan(L, nt, nph, minc=minc, max_levels=nlev)
    o = oracle.Plan(L, nt, nph, minc=minc)
    ins = workload.nl_inputs(L, nlev, 9, minc=minc)
    rad = radial(nlev)
    lcut = [L] * nlev
    dev = torch.device("cuda")
    tin = [torch.from_numpy(x).to(dev) for x in ins]
    outs = [torch.zeros((nlev, p.lm_max), dtype=torch.complex128, device=dev) for _ in range(10)]
    grids = torch.zeros((nlev, 18, nph, nt), dtype=torch.float64, device=dev)
    sht.nl_step(p, tin, outs, *rad, lcut, grids=grids)
    got = [x.cpu().numpy() for x in outs]
    sht.nl_step(p, tin, outs, *rad, lcut)
    want_g, want = oracle_step(o, ins, *rad, lcut)
    for k in range(10):
        assert rel_l2(got[k], want[k]) < TOL, sht.NL_OUTPUTS[k]
        assert np.array_equal(got[k], outs[k].cpu().numpy()), sht.NL_OUTPUTS[k]
    for k in range(18):
        assert rel_l2(grids[:, k].cpu().numpy(), want_g[:, k]) < TOL, sht.NL_GRIDS[k]
    p.close()


# the radial loop's grid stage: slots of 2, 4, 16 and 32 lanes, block-wide
# passes (n_phi = 160), under the switches of every dump of the reference
@pytest.mark.parametrize("case", rc.CASES)
@pytest.mark.parametrize("L,nt,nph", [(15, 24, 48), (15, 28, 96), (20, 36, 160), (30, 44, 384), (20, 36, 768)])
def test_rloop_matches_oracle(case, L, nt, nph):
    """Two interior levels, one cut below l_max, against the oracle's radial
    loop.  The Courant steps and explicit terms are held to 1e-11, the bar of
    the loop's comparison at l_max = 255: the Lorentz force and the Coriolis
    terms of the dumps' parameters cancel a few digits."""
    from oracle import oracle
    from rloop_reference import oracle_rloop
    nlev = 2
    ph = rc.phys_of(rc.load(case))
    print("rloop", case, L, nt, nph, flush=True)
    ins = workload.nl_inputs(L, nlev, stream=13)
    fields = {n: None for n in sht.RLOOP_IN}
    fields.update(dict(zip(sht.NL_INPUTS, ins)))
    fields["xi"] = np.stack([workload.coefficients(L, 13, 20, i, potential=False) for i in range(nlev)])
    fields["phi"] = np.stack([workload.coefficients(L, 13, 21, i, potential=False) for i in range(nlev)])
    r = np.array([0.8, 1.2])
    one = np.ones(nlev)
    rad = {"r": r, "or1": 1 / r, "or2": 1 / r ** 2, "or4": 1 / r ** 4, "orho1": 1 / (1 + 0.1 * r),
           "beta": -0.1 / (1 + 0.1 * r), "otemp1": 1 / (1.5 - 0.2 * r), "visc": one, "lambda": 1 + 0.1 * r,
           "temp0": one, "epscProf": one, "delxr2": np.full(nlev, 1e-3), "delxh2": np.full(nlev, 2e-2),
           "nR": np.array([5, 9], dtype=np.int32), "l_R": np.array([L, L - 2], dtype=np.int32)}
    names = rc.outputs_of(dict(ph, **{k: ph.get(k, 0) for k in sht.RLOOP_INT}))
    p = sht.Plan(L, nt, nph, max_levels=nlev)
    outs = {n: np.zeros((nlev, p.lm_max), dtype=np.complex128) for n in names}
    dtr, dth = np.zeros(nlev), np.zeros(nlev)
    sht.rloop(p, ph, nlev, rad, fields, outs, dtr, dth)
    p.close()
    o = oracle.Plan(L, nt, nph)
    want, wtr, wth = oracle_rloop(o, ph, nlev, rad, fields, 1)
    for n in names:
        assert rel_l2(outs[n], want[n]) < 1e-11, n
    assert rel_l2(dtr, wtr) < 1e-11 and rel_l2(dth, wth) < 1e-11
