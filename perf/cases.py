"""The transform work a user of this package runs, as timed cases: the calls of
module sht on host arrays, the batched transforms, the nonlinear step in its
precisions, the radial loop with its physics switches, and batches of uneven
transform jobs.

A case is a dict of plain values; ``call`` names the entry point.  Grids
follow the package's own sizing (``workload.grid_size``), inputs the spectra
of its workloads: fields of amplitude l^-5/3 with random phases.
"""
import functools
import math

import numpy as np
import torch

from magic_amd import sht, workload

# truncations whose grid sizes have small factors only, as runs choose them
# (l_max: 3/2 rule, n_phi = 2^i 3^j 5^k); odd and even, powers of two,
# multiples of 3 and of 5 among the grids
TRUNCATIONS = (31, 42, 53, 64, 85, 106, 127, 128, 133, 159, 170, 191, 213, 255, 256, 319, 341, 383, 426, 511)

FIELDS = sht.NL_INPUTS
PRECISIONS = {"fp64": sht.PREC_FP64, "split": sht.PREC_SPLIT16, "split_rec": sht.PREC_SPLIT16_REC}

# physics switches of the radial loop, as the runs of the test suite use them
_CONVECTION = dict(l_conv=1, l_conv_nl=1, l_heat=1, l_heat_nl=1, l_corr=1, CorFac=1000.0, oek=1000.0,
                   opm=0.2, courfac=2.5, alffac=1.0, epsc=0.5)
_DYNAMO = dict(_CONVECTION, l_mag=1, l_mag_LF=1, l_mag_nl=1, l_cour_alf_damp=1, LFfac=200.0)
SWITCHES = {
    "mhd_curl": dict(_DYNAMO, l_adv_curl=1),
    "mhd_ugradu": dict(_DYNAMO, l_adv_curl=0),
    "anelastic_mhd": dict(_DYNAMO, l_adv_curl=0, l_anel=1, ViscHeatFac=0.02, OhmLossFac=0.05),
    "double_diffusion": dict(_CONVECTION, l_adv_curl=1, l_chemical_conv=1, epscXi=0.25),
}


def listed():
    return [
        # one radial level through module sht as the Fortran program calls it:
        # host arrays in, host grids out, at the size of the benchmark samples
        dict(name="level_synthesis_l64", call="level_synthesis", l_max=64, minc=1),
        # the forward call of one level of a production-size run
        dict(name="level_analysis_l255", call="level_analysis", l_max=255, minc=1),
        # batched transforms of device arrays: post-processing, initial fields;
        # a grid of 160 x 320 and an odd number of levels
        dict(name="synthesis_l106x41", call="synthesis", l_max=106, minc=1, nlev=41),
        # forward, the power-of-two grid 256 x 512
        dict(name="analysis_l170x65", call="analysis", l_max=170, minc=1, nlev=65),
        # the nonlinear step of the benchmark sample's size (fourfold symmetry)
        dict(name="step_fp64_l64x33_minc4", call="step", l_max=64, minc=4, nlev=33, precision="fp64"),
        # an ordinary resolution on a power-of-two grid
        dict(name="step_fp64_l170x65", call="step", l_max=170, minc=1, nlev=65, precision="fp64"),
        # the headline workload in the default precision ...
        dict(name="step_fp64_l255x97", call="step", l_max=255, minc=1, nlev=97, precision="fp64"),
        # ... and in the split precision
        dict(name="step_split_l255x97", call="step", l_max=255, minc=1, nlev=97, precision="split"),
        # high resolution, stored split tables
        dict(name="step_split_l511x32", call="step", l_max=511, minc=1, nlev=32, precision="split"),
        # a time-step stage of a dynamo as the Fortran plugin hands it over: host arrays
        dict(name="radial_loop_mhd_l64x31_host", call="radial_loop", l_max=64, minc=4, nlev=31,
             precision="fp64", switches="mhd_curl", host=True),
        # a dynamo run with u.grad u advection, fields resident on the GPU
        dict(name="radial_loop_ugradu_l255x97", call="radial_loop", l_max=255, minc=1, nlev=97,
             precision="fp64", switches="mhd_ugradu", host=False),
        # uneven independent transform jobs in one batch
        dict(name="jobs_16", call="jobs", njobs=16, batch=3),
    ]


def draw(rng):
    call = rng.choice(["level_synthesis", "level_analysis", "synthesis", "analysis", "step", "step", "step",
                       "radial_loop", "radial_loop", "jobs"])
    if call == "jobs":
        return dict(call=call, njobs=rng.randint(2, 16), batch=rng.randint(1, 10 ** 6))
    top = 255 if call == "radial_loop" else 511
    l_max = rng.choice([l for l in TRUNCATIONS if l <= top])
    minc = rng.choice([m for m in (1, 1, 1, 2, 4) if _fits(l_max, m)])
    case = dict(call=call, l_max=l_max, minc=minc)
    if call.startswith("level"):
        return case
    # levels up to 97, and no more work than the headline step
    most = max(2, min(97, int(97 * minc * (255 / l_max) ** 3)))
    case["nlev"] = int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    if call == "step":
        case["precision"] = rng.choice(["fp64", "split"] if l_max <= 255 else ["fp64", "split", "split_rec"])
    if call == "radial_loop":
        case["switches"] = rng.choice(sorted(SWITCHES))
        case["precision"] = rng.choice(["fp64", "fp64", "split"])
        case["host"] = l_max <= 85 and rng.random() < 0.5
    return case


def _fits(l_max, minc):
    try:
        workload.grid_size(l_max, 20, minc)
    except ValueError:
        return False
    return True


# ------------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=4)
def _degrees(l_max, minc):
    l, m = workload.lm_index(l_max, None, minc)
    dev = _device()
    return torch.from_numpy(l).to(dev), torch.from_numpy(m).to(dev)


def _coefficients(gen, l_max, minc, shape, power):
    """Random phases, amplitude l^-5/3 divided by l^power; real at m = 0,
    zero at l = 0 for potentials (power > 0)."""
    l, m = _degrees(l_max, minc)
    d = l.clamp(min=1).double()
    amp = d ** (-5.0 / 3.0)
    if power == 2:
        amp = amp / (d * (d + 1.0))
    elif power == 1:
        amp = amp / d
    if power:
        amp = torch.where(l == 0, 0.0, amp)
    phase = torch.rand(tuple(shape) + (l.numel(),), generator=gen, dtype=torch.float64, device=l.device)
    c = torch.polar(amp.expand_as(phase).contiguous(), 2.0 * math.pi * phase)
    return torch.where(m == 0, c.real + 0j, c)


# the l-factor each transform applies to the potential
_POWER = {"w": 2, "b": 2, "s": 0, "xi": 0}


def _fields(gen, case, names):
    return {n: _coefficients(gen, case["l_max"], case["minc"], (case["nlev"],), _POWER.get(n, 1)) for n in names}


def _generator(seed):
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(seed))
    return gen


def _radial(case):
    """Per-level factors of a shell between radii 0.55 and 1.45, weakly
    stratified where the switches are anelastic."""
    n = case["nlev"]
    r = np.linspace(0.55, 1.45, n) if n > 1 else np.array([1.0])
    one = np.ones(n)
    anel = case.get("switches") == "anelastic_mhd"
    rho = 1.0 / (1.0 + 0.1 * r) if anel or case["call"] == "step" else one
    return {"r": r, "or1": 1 / r, "or2": 1 / r ** 2, "or4": 1 / r ** 4, "orho1": rho,
            "beta": -0.1 * rho if anel else 0 * one, "otemp1": 1 / (1.5 - 0.2 * r) if anel else one,
            "visc": one, "lambda": 1 + 0.1 * r if anel else one, "temp0": one, "epscProf": one,
            "delxr2": np.full(n, 1e-3), "delxh2": np.full(n, 2e-2),
            "nR": np.arange(2, n + 2, dtype=np.int32), "l_R": np.full(n, case["l_max"], dtype=np.int32)}


def _loop_fields(case):
    ph = SWITCHES[case["switches"]]
    names = list(FIELDS[:5]) + ["s"]
    if ph.get("l_chemical_conv"):
        names.append("xi")
    if ph.get("l_mag"):
        names += FIELDS[6:]
    return names


def _loop_outputs(case):
    ph = SWITCHES[case["switches"]]
    names = ["dwdt", "dzdt", "dpdt", "dsdt", "dVSrLM"]
    if ph.get("l_chemical_conv"):
        names += ["dxidt", "dVXirLM"]
    if ph.get("l_mag"):
        names += ["dbdt", "djdt", "dVxBhLM"]
    return names


def _job_specs(case):
    """(l_max, kind, fields, levels) of the jobs of one batch."""
    return [(L, kind, nf, max(3, nlev // 2))
            for L, kind, nf, nlev in workload.batch_specs(case["njobs"], case["batch"])]


def _job_inputs(gen, spec):
    L, kind, nf, nlev = spec
    if kind == sht.JOB_SCALAR:
        return _coefficients(gen, L, 1, (1, nf, nlev), 0)
    return torch.cat([_coefficients(gen, L, 1, (1, nf, nlev), p) for p in (2, 1, 1)])


def _grids(gen, case):
    """A vector field on the grid, (n_phi, n_theta) or (nlev, n_phi, n_theta):
    random modes falling as k^-5/3 in latitude and longitude, the horizontal
    components times sin(theta)."""
    n_theta, n_phi = workload.grid_size(case["l_max"], 20, case["minc"])
    lead = (case["nlev"],) if "nlev" in case else ()
    kp = torch.fft.fftfreq(n_phi, 1.0 / n_phi, dtype=torch.float64, device=gen.device)[:, None]
    kt = torch.fft.rfftfreq(n_theta, 1.0 / n_theta, dtype=torch.float64, device=gen.device)
    amp = (1.0 + kp * kp + kt * kt) ** (-5.0 / 6.0)
    sin = torch.sin((torch.arange(n_theta, dtype=torch.float64, device=gen.device) + 0.5) * (math.pi / n_theta))
    # rows alternate theta_k, pi - theta_k
    north = torch.arange(n_theta // 2, device=gen.device)
    rows = torch.stack([north, n_theta - 1 - north], 1).reshape(-1)
    out = []
    for comp in range(3):
        x = torch.randn(lead + (n_phi, n_theta // 2 + 1, 2), generator=gen, dtype=torch.float64, device=gen.device)
        g = torch.fft.irfft2(torch.view_as_complex(x) * amp, s=(n_phi, n_theta), norm="ortho")
        out.append((g if comp == 0 else g * sin)[..., rows].contiguous())
    return out


def _plan(case):
    n_theta, n_phi = workload.grid_size(case["l_max"], 20, case["minc"])
    return sht.Plan(case["l_max"], n_theta, n_phi, minc=case["minc"],
                    precision=PRECISIONS[case.get("precision", "fp64")], max_levels=case.get("nlev", 1))


def _level_inputs(case, seed):
    gen = _generator(seed)
    if case["call"] in ("level_synthesis", "synthesis"):
        lead = (case["nlev"],) if "nlev" in case else ()
        return [_coefficients(gen, case["l_max"], case["minc"], lead, p) for p in (2, 1, 1)]
    return _grids(gen, case)


def prepare(case, seed):
    call = case["call"]
    if call == "jobs":
        gen = _generator(seed)
        jobs = []
        for spec in _job_specs(case):
            x = _job_inputs(gen, spec)
            jobs.append((spec[0], spec[1], x, torch.zeros_like(x)))
        torch.cuda.synchronize()
        return {"call": call, "jobs": jobs, "batch": sht.Batch(jobs), "stream": torch.cuda.Stream()}
    state = {"call": call, "plan": _plan(case)}
    if call in ("level_synthesis", "level_analysis"):
        state["inputs"] = [x.cpu().numpy() for x in _level_inputs(case, seed)]
        state["lcut"] = case["l_max"]
        return state
    nlev, plan = case["nlev"], state["plan"]
    coef = lambda: torch.zeros((nlev, plan.lm_max), dtype=torch.complex128, device="cuda")  # noqa: E731
    if call in ("synthesis", "analysis"):
        state["inputs"] = _level_inputs(case, seed)
        state["lcut"] = [case["l_max"]] * nlev
        grid = lambda: torch.zeros((nlev, plan.n_phi, plan.n_theta), dtype=torch.float64, device="cuda")  # noqa: E731
        state["outputs"] = [grid() if call == "synthesis" else coef() for _ in range(3)]
        torch.cuda.synchronize()
        return state
    state["radial"] = _radial(case)
    gen = _generator(seed)
    if call == "step":
        state["inputs"] = list(_fields(gen, case, FIELDS).values())
        state["outputs"] = [coef() for _ in range(10)]
        state["lcut"] = [case["l_max"]] * nlev
        # steps are issued on a side stream and return without waiting
        state["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
        return state
    fields = _fields(gen, case, _loop_fields(case))
    outputs = {n: coef() for n in _loop_outputs(case)}
    if case["host"]:
        fields = {n: x.cpu().numpy() for n, x in fields.items()}
        outputs = {n: x.cpu().numpy() for n, x in outputs.items()}
    state.update(fields=fields, outputs=outputs, switches=SWITCHES[case["switches"]], nlev=nlev,
                 dtrkc=np.zeros(nlev), dthkc=np.zeros(nlev))
    torch.cuda.synchronize()
    return state


def run(state):
    call = state["call"]
    if call == "jobs":
        state["batch"].execute(stream=state["stream"])
        return [job[3] for job in state["jobs"]]
    plan = state["plan"]
    if call == "level_synthesis":
        return plan.torpol_to_spat(*state["inputs"], state["lcut"])
    if call == "level_analysis":
        return plan.spat_to_qst(*state["inputs"], state["lcut"])
    if call == "synthesis":
        plan.torpol_to_spat_batch(*state["inputs"], state["lcut"], *state["outputs"])
        return state["outputs"]
    if call == "analysis":
        plan.spat_to_qst_batch(*state["inputs"], state["lcut"], *state["outputs"])
        return state["outputs"]
    r = state["radial"]
    if call == "step":
        sht.nl_step(plan, state["inputs"], state["outputs"], r["or2"], r["or4"], r["orho1"], 0.8,
                    state["lcut"], stream=state["stream"])
        return state["outputs"]
    sht.rloop(plan, state["switches"], state["nlev"], r, state["fields"], state["outputs"], state["dtrkc"],
              state["dthkc"])
    return {**state["outputs"], "dtrkc": state["dtrkc"], "dthkc": state["dthkc"]}


# --------------------------------------------------------------------- work
def _transform_flops(case, scalars, vectors, products=0):
    """Flops of transforming so many scalar and vector fields of one level:
    one complex Legendre sum per component with the equatorial symmetry, one
    real FFT per theta row and component, and the products per grid point."""
    n_theta, n_phi = workload.grid_size(case["l_max"], 20, case["minc"])
    ncoef = _degrees(case["l_max"], case["minc"])[0].numel()
    comps = scalars + 3 * vectors
    return (4.0 * (n_theta // 2) * ncoef * comps + 2.5 * n_phi * math.log2(n_phi) * n_theta * comps +
            float(products) * n_theta * n_phi)


def work(case):
    call = case["call"]
    if call == "jobs":
        nbytes = flops = 0.0
        for L, kind, nf, nlev in _job_specs(case):
            comps = 3 if kind == sht.JOB_VECTOR else 1
            nbytes += 2 * 16.0 * comps * nf * nlev * ((L + 1) * (L + 2) // 2)
            n = 3 * (L + 1) // 2
            flops += 2.0 * comps * nf * nlev * (4.0 * (n // 2) * ((L + 1) * (L + 2) // 2) +
                                                2.5 * 2 * n * math.log2(2 * n) * n)
        return {"bytes": nbytes, "flops": flops}
    n_theta, n_phi = workload.grid_size(case["l_max"], 20, case["minc"])
    coef = 16.0 * _degrees(case["l_max"], case["minc"])[0].numel()
    nlev = case.get("nlev", 1)
    if call in ("level_synthesis", "level_analysis", "synthesis", "analysis"):
        return {"bytes": nlev * 3 * (coef + 8.0 * n_theta * n_phi), "flops": nlev * _transform_flops(case, 0, 1)}
    if call == "step":
        # u, curl u, B, curl B, s and its gradient; Adv, V s, V x B, u.grad s
        return {"bytes": nlev * 21 * coef, "flops": nlev * _transform_flops(case, 4, 7, 70)}
    ph = SWITCHES[case["switches"]]
    mag, chem = bool(ph.get("l_mag")), bool(ph.get("l_chemical_conv"))
    scalars = 1 + chem + (5 if not ph["l_adv_curl"] else 0) + bool(ph.get("l_anel"))
    vectors = 2 + 2 * mag + 1 + 1 + chem + mag
    fields = len(_loop_fields(case)) + len(_loop_outputs(case))
    return {"bytes": nlev * fields * coef, "flops": nlev * _transform_flops(case, scalars, vectors, 100)}


# ---------------------------------------------- the same in plain 64-bit torch
class _Transform:
    """Spherical-harmonic transforms of one truncation by dense Legendre sums
    and torch.fft, all in float64: orthonormal P_lm without the Condon-Shortley
    phase, rows alternating theta_k, pi - theta_k, vectors times sin(theta)."""

    def __init__(self, l_max, minc):
        self.L, self.minc = l_max, minc
        self.nt, self.nph = workload.grid_size(l_max, 20, minc)
        dev = _device()
        x, wt = self._gauss(self.nt)
        half = self.nt // 2
        rows = np.empty(self.nt, np.longdouble)
        rows[0::2], rows[1::2] = x[:half], -x[:half]
        w = np.repeat(wt[:half], 2)
        self.x = torch.from_numpy(rows.astype(np.float64)).to(dev)
        self.sin = torch.from_numpy(np.sqrt((1 - rows) * (1 + rows)).astype(np.float64)).to(dev)
        self.w = torch.from_numpy((w * 2 * np.longdouble(math.pi)).astype(np.float64)).to(dev)
        self.osin2 = 1.0 / self.sin ** 2
        self.l, self.m = _degrees(l_max, minc)
        self.ll = (self.l * (self.l + 1)).double()
        self.orders = list(range(0, l_max + 1, minc))
        self._tables()

    @staticmethod
    def _gauss(n):
        k = np.arange(1, n + 1, dtype=np.longdouble)
        z = np.cos(np.longdouble(math.pi) * (k - 0.25) / (n + np.longdouble(0.5)))
        for _ in range(8):
            p1, p2 = np.ones_like(z), np.zeros_like(z)
            for j in range(1, n + 1):
                p1, p2 = ((2 * j - 1) * z * p1 - (j - 1) * p2) / j, p1
            dp = n * (z * p1 - p2) / (z * z - 1)
            z = z - p1 / dp
        return z, 2 / ((1 - z * z) * dp * dp)

    def _tables(self):
        """P[l] of every order at once: (n_m, n_theta) per degree."""
        dev, L = self.x.device, self.L
        m = torch.tensor(self.orders, dtype=torch.float64, device=dev)[:, None]
        k = np.arange(1, L + 1, dtype=np.float64)
        norm = np.concatenate([[0.0], np.cumsum(0.5 * np.log1p(1.0 / (2.0 * k)))]) - 0.5 * math.log(4 * math.pi)
        pmm = torch.exp(torch.from_numpy(norm[self.orders]).to(dev)[:, None] + m * torch.log(self.sin)[None, :])
        eps = lambda l: torch.sqrt(((l * l - m * m) / (4.0 * l * l - 1.0)).clamp(min=0.0))  # noqa: E731
        self.P = torch.zeros((L + 2, len(self.orders), self.nt), dtype=torch.float64, device=dev)
        p, pm = torch.zeros_like(pmm), torch.zeros_like(pmm)
        for l in range(L + 2):
            p = torch.where(m == l, pmm, p)
            self.P[l] = p
            e1 = eps(float(l + 1))
            nxt = torch.where(m <= l, (self.x * p - eps(float(l)) * pm) / torch.where(e1 > 0, e1, 1.0), 0.0)
            p, pm = nxt, p

    def _order(self, mc):
        """(slice of lm, P, sin dP/dtheta) of one order: tables (n_theta, n_l)."""
        m, L = self.orders[mc], self.L
        start = sum(L - k + 1 for k in self.orders[:mc])
        l = torch.arange(m, L + 1, dtype=torch.float64, device=self.x.device)
        e = lambda d: torch.sqrt((d * d - m * m) / (4.0 * d * d - 1.0))  # noqa: E731
        P = self.P[m:L + 1, mc].T
        up = self.P[m + 1:L + 2, mc].T
        low = torch.cat([torch.zeros_like(P[:, :1]), P[:, :-1]], 1)
        return slice(start, start + L - m + 1), P, l * e(l + 1) * up - (l + 1) * e(l) * low

    def _to_fourier(self, terms, nout):
        """terms: (output, table 0 P / 1 dP, coefficients (nlev, lm))."""
        nlev = terms[0][2].shape[0]
        F = torch.zeros((nout, nlev, self.nt, self.nph // 2 + 1), dtype=torch.complex128, device=self.x.device)
        for mc in range(len(self.orders)):
            s, P, dP = self._order(mc)
            for o, tab, c in terms:
                v = c[:, s]
                cols = torch.cat([v.real, v.imag]).contiguous()
                y = ((dP if tab else P) @ cols.T.contiguous()).T
                F[o, :, :, mc] += torch.complex(y[:nlev].contiguous(), y[nlev:].contiguous())
        return [torch.fft.irfft(f, n=self.nph, dim=-1, norm="forward") for f in F]

    def scalar(self, s):
        return self._to_fourier([(0, 0, s)], 1)[0]

    def gradient(self, s):
        return self._to_fourier([(0, 1, s), (1, 0, 1j * self.m * s)], 2)

    def sphtor(self, S, T):
        return self._to_fourier([(0, 1, S), (0, 0, 1j * self.m * T), (1, 0, 1j * self.m * S), (1, 1, -T)], 2)

    def torpol(self, W, dW, Z):
        return [self.scalar(self.ll * W)] + self.sphtor(dW, Z)

    def curl(self, or2, B, ddB, J, dJ):
        return [self.scalar(self.ll * J)] + self.sphtor(dJ, or2[:, None] * self.ll * B - ddB)

    def _from_grids(self, terms, grids, nout):
        """terms: (output, table 0 P / 1 dP, grid, sign, whether times i m)."""
        F = [torch.fft.rfft(g, dim=-1, norm="forward") for g in grids]
        nlev = grids[0].shape[0]
        out = torch.zeros((nout, nlev, self.l.numel()), dtype=torch.complex128, device=self.x.device)
        for mc, m in enumerate(self.orders):
            s, P, dP = self._order(mc)
            for o, tab, g, sign, im in terms:
                f = F[g][:, :, mc] * self.w
                rows = torch.cat([f.real, f.imag]).contiguous()
                y = rows @ (dP if tab else P).contiguous()
                y = sign * torch.complex(y[:nlev].contiguous(), y[nlev:].contiguous())
                out[o][:, s] += 1j * m * y if im else y
        return list(out)

    def to_scalar(self, f):
        return self._from_grids([(0, 0, 0, 1, False)], [f], 1)[0]

    def to_qst(self, f, vt, vp):
        """f, vt, vp grids (nlev, n_theta, n_phi) to Q, S, T."""
        o2 = self.osin2[:, None]
        q, s, t = self._from_grids([(0, 0, 0, 1, False), (1, 1, 1, 1, False), (1, 0, 2, -1, True),
                                    (2, 1, 2, -1, False), (2, 0, 1, -1, True)], [f, vt * o2, vp * o2], 3)
        oll = 1.0 / self.ll.clamp(min=1.0)
        return q, s * oll, t * oll


@functools.lru_cache(maxsize=1)
def _transform(l_max, minc):
    return _Transform(l_max, minc)


def _column(v, dev):
    return torch.from_numpy(np.asarray(v, dtype=np.float64)).to(dev)[:, None, None]


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def _exact_step(case, f):
    t = _transform(case["l_max"], case["minc"])
    rad = _radial(case)
    dev = t.x.device
    or2v = torch.from_numpy(rad["or2"]).to(dev)
    or2, or4, orho1 = (_column(rad[k], dev) for k in ("or2", "or4", "orho1"))
    o2 = t.osin2[:, None]
    u = t.torpol(f["w"], f["dw"], f["z"])
    cu = t.curl(or2v, f["w"], f["ddw"], f["z"], f["dz"])
    fac = [o2, or4, or4]
    adv = [-c * x for c, x in zip(fac, _cross(cu, u))]
    del cu
    b = t.torpol(f["b"], f["db"], f["aj"])
    cb = t.curl(or2v, f["b"], f["ddb"], f["aj"], f["dj"])
    adv = [a + 0.8 * c * x for a, c, x in zip(adv, fac, _cross(cb, b))]
    del cb
    vxb = [orho1 * c * x for c, x in zip(fac, _cross(u, b))]
    del b
    s = t.scalar(f["s"])
    st, sp = t.gradient(f["s"])
    vs = [u[0] * s, or2 * u[1] * s, or2 * u[2] * s]
    ugs = or2 * o2 * (u[1] * st + u[2] * sp)
    del u, s, st, sp
    return [*t.to_qst(*adv), *t.to_qst(*vs), *t.to_qst(*vxb), t.to_scalar(ugs)]


def _exact_loop(case, f):
    ph = SWITCHES[case["switches"]]
    t = _transform(case["l_max"], case["minc"])
    rad = _radial(case)
    dev = t.x.device
    or2v = torch.from_numpy(rad["or2"]).to(dev)
    r, or1, or2, or4, orho1, beta, otemp1, visc, lam = (
        _column(rad[k], dev) for k in ("r", "or1", "or2", "or4", "orho1", "beta", "otemp1", "visc", "lambda"))
    o2 = t.osin2[:, None]
    cosn2 = t.x[:, None] * o2
    mag, anel = bool(ph.get("l_mag")), bool(ph.get("l_anel"))
    fac = [o2, or4, or4]
    u = t.torpol(f["w"], f["dw"], f["z"])
    vr, vt, vp = u
    if ph["l_adv_curl"]:
        cu = t.curl(or2v, f["w"], f["ddw"], f["z"], f["dz"])
        adv = [-c * x for c, x in zip(fac, _cross(cu, u))]
    else:
        cvr = t.scalar(t.ll * f["z"])
        dr = t.torpol(f["dw"], f["ddw"], f["dz"])
        gt, gp = t.gradient(t.ll * f["w"])
        tp, pp = (o2 * x for x in t.sphtor(1j * t.m * f["dw"], 1j * t.m * f["z"]))
        adv = [-or2 * orho1 * (vr * (dr[0] - (2 * or1 + beta) * vr) + o2 * (vt * (gt - r * vt) + vp * (gp - r * vp))),
               or4 * orho1 * (-vr * (dr[1] - beta * vt) + vt * (cosn2 * vt + pp + dr[0]) + vp * (cosn2 * vp - tp)),
               or4 * orho1 * (-vr * (dr[2] - beta * vp) - vt * (tp + cvr) - vp * pp)]
    vr2 = or4 * ph["courfac"] ** 2 * (orho1 * vr) ** 2
    vh2 = or2 * ph["courfac"] ** 2 * (vt ** 2 + vp ** 2) * o2 * orho1 ** 2
    out = {}
    heat = None
    if anel:
        t1 = dr[0] - (2 * or1 + beta) * vr
        t2 = cosn2 * vt + pp + dr[0] - or1 * vr
        t3 = pp + cosn2 * vt + or1 * vr
        t6 = 2 * tp + cvr - 2 * cosn2 * vp
        t4 = r * dr[1] - (2 + beta * r) * vt + or1 * gt
        t5 = r * dr[2] - (2 + beta * r) * vp + or1 * gp
        heat = ph["ViscHeatFac"] * or4 * orho1 * otemp1 * visc * (
            2 * t1 ** 2 + 2 * t2 ** 2 + 2 * t3 ** 2 + t6 ** 2 + o2 * (t4 ** 2 + t5 ** 2) - 2 / 3 * (beta * vr) ** 2)
    ll = t.ll
    if mag:
        b = t.torpol(f["b"], f["db"], f["aj"])
        cb = t.curl(or2v, f["b"], f["ddb"], f["aj"], f["dj"])
        adv = [a + ph["LFfac"] * c * x for a, c, x in zip(adv, fac, _cross(cb, b))]
        if anel:
            heat = heat + ph["OhmLossFac"] * or2 * otemp1 * lam * (or2 * cb[0] ** 2 + o2 * (cb[1] ** 2 + cb[2] ** 2))
        damp = (0.5 * (1 + ph["opm"])) ** 2
        ar = b[0] ** 2 * ph["LFfac"] * orho1
        ah = (b[1] ** 2 + b[2] ** 2) * ph["LFfac"] * o2 * orho1
        vr2 = vr2 + or4 * ph["alffac"] ** 2 * ar ** 2 / (ar + damp / _column(rad["delxr2"], dev))
        vh2 = vh2 + or2 * ph["alffac"] ** 2 * ah ** 2 / (ah + damp / _column(rad["delxh2"], dev))
        q, s, x = t.to_qst(*[orho1 * c * x for c, x in zip(fac, _cross(u, b))])
        out["djdt"] = ll * or4[:, 0] * q
        out["dVxBhLM"] = -ll * r[:, 0] ** 2 * s
        out["dbdt"] = ll * x
    for name, v, dx in (("dtrkc", vr2, rad["delxr2"]), ("dthkc", vh2, rad["delxh2"])):
        out[name] = np.minimum(1e10, np.sqrt(dx / v.amax(dim=(1, 2)).cpu().numpy()))
    scalars = [("s", "dVSrLM", "dsdt", ph["epsc"] * rad["epscProf"])]
    if ph.get("l_chemical_conv"):
        scalars.append(("xi", "dVXirLM", "dxidt", ph["epscXi"] * np.ones(case["nlev"])))
    for name, radial, rate, mean in scalars:
        s = t.scalar(f[name])
        out[radial], st, _ = t.to_qst(vr * s, or2 * vt * s, or2 * vp * s)
        out[rate] = ll * st
        out[rate][:, 0] = torch.from_numpy(mean).to(dev)
    if anel:
        out["dsdt"] = out["dsdt"] + t.to_scalar(heat)
    advr, advt, advp = t.to_qst(*adv)
    # Coriolis terms: neighbours l - 1 and l + 1 of the same order
    l, m = t.l.double(), t.m.double()
    e = lambda d: torch.sqrt(((d * d - m * m) / (4 * d * d - 1)).clamp(min=0.0))  # noqa: E731
    cS, cA = e(l), e(l + 1)

    def below(x):
        return torch.where(t.l > t.m, torch.roll(x, 1, 1), 0)

    def above(x):
        return torch.where(t.l < t.L, torch.roll(x, -1, 1), 0)
    c2, im = 2.0 * ph["CorFac"], 1j * m
    o1, q2 = or1[:, 0], or2[:, 0]
    w, dw, z = f["w"], f["dw"], f["z"]
    out["dwdt"] = q2 * advr + c2 * o1 * (im * dw - (l - 1) * cS * below(z) + (l + 2) * cA * above(z))
    out["dzdt"] = ll * advp + c2 * q2 * (
        im * z + (l * l - 1) * cS * below(dw) - o1 * (l + 1) * cS * (l - 1) * l * below(w) +
        l * (l + 2) * cA * above(dw) + o1 * l * cA * (l + 1) * (l + 2) * above(w))
    out["dpdt"] = -ll * advt + c2 * q2 * (-im * (dw + o1 * ll * w) + (l * l - 1) * cS * below(z) +
                                          l * (l + 2) * cA * above(z))
    out["dpdt"][:, 0] = 0
    return out


def exact(case, seed):
    call = case["call"]
    gen = _generator(seed)
    if call == "jobs":
        # the round trip of a band-limited field is the identity (vector jobs:
        # Q = l(l+1) W, S = dW, T = Z, the horizontal parts zero at l = 0)
        out = []
        for spec in _job_specs(case):
            x = _job_inputs(gen, spec)
            if spec[1] == sht.JOB_VECTOR:
                l = _degrees(spec[0], 1)[0]
                x = torch.cat([x[:1] * (l * (l + 1)).double(), torch.where(l == 0, 0, x[1:])])
            out.append(x)
        return out
    if call in ("step", "radial_loop"):
        f = _fields(gen, case, FIELDS if call == "step" else _loop_fields(case))
        return _exact_step(case, f) if call == "step" else _exact_loop(case, f)
    t = _transform(case["l_max"], case["minc"])
    one = "nlev" not in case
    x = [v[None] if one else v for v in _level_inputs(case, seed)]
    if call in ("level_synthesis", "synthesis"):
        out = [g.transpose(1, 2).contiguous() for g in t.torpol(*x)]
    else:
        out = list(t.to_qst(*[g.transpose(1, 2) for g in x]))
    return tuple(v[0] for v in out) if one else out
