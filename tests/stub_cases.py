"""Scenarios of the library's host code on the stand-in runtime of
hip_stub.cpp, one per process: python stub_cases.py STUB LIBRARY SCENARIO."""
import ctypes
import os
import sys

import numpy as np

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from magic_amd import sht  # noqa: E402

FP64, SPLIT16, SPLIT16_REC = 0, 1, 2
# a plan of each kind at its smallest: l_max, minc, n_theta, n_phi
PLANS = {FP64: (16, 1, 32, 64), SPLIT16: (16, 1, 32, 64), SPLIT16_REC: (256, 16, 16, 64)}


class Stub:
    def __init__(self, stub, library):
        self.s = ctypes.CDLL(stub, mode=ctypes.RTLD_GLOBAL)
        self.s.stub_log.restype = ctypes.c_char_p
        self.s.stub_fail.argtypes = [ctypes.c_long]
        self.s.stub_bytes.restype = self.s.stub_live.restype = ctypes.c_size_t
        self.L = ctypes.CDLL(library)
        self.L.mhx_last_error.restype = ctypes.c_char_p
        sht._lib = self.L

    def log(self):
        return [x.split() for x in self.s.stub_log().decode().splitlines()]

    def plan(self, precision, levels=2, shape=None):
        l_max, minc, nt, nph = shape or PLANS[precision]
        h = ctypes.c_void_p()
        rc = self.L.mhx_plan_create(l_max, 0, minc, nt, nph, precision, levels, ctypes.byref(h))
        assert rc == 0, self.L.mhx_last_error()
        lm = ctypes.c_int()
        self.L.mhx_plan_info(h, ctypes.byref(lm), None, None, None)
        return Handle(self, h, lm.value, l_max, nt, nph)


class Handle:
    def __init__(self, stub, h, lm_max, l_max, nt, nph):
        self.stub, self.L, self.h = stub, stub.L, h
        self.lm_max, self.l_max, self.nt, self.nph = lm_max, l_max, nt, nph

    def close(self):
        self.L.mhx_plan_destroy(self.h)

    def host(self, n):
        return (ctypes.c_double * int(n))()

    def call(self, name):
        """one call on host arrays; its return code"""
        c, g, L = self.host(2 * self.lm_max), [self.host(self.nt * self.nph) for _ in range(3)], self.L
        a = self.host(2 * (self.l_max + 1))
        t = self.host(self.nt // 2 * self.lm_max)
        z = ctypes.c_double
        return {"axi_to_spat": lambda: L.mhx_axi_to_spat(self.h, a, g[0]),
                "toraxi_to_spat": lambda: L.mhx_toraxi_to_spat(self.h, a, g[0], g[1], self.l_max),
                "tables": lambda: L.mhx_plan_tables(self.h, None, None, t, t),
                "scal_to_spat": lambda: L.mhx_scal_to_spat(self.h, c, g[0], self.l_max),
                "spat_to_qst": lambda: L.mhx_spat_to_qst(self.h, *g, c, self.host(2 * self.lm_max),
                                                         self.host(2 * self.lm_max), self.l_max)}[name]()

    def step(self, nlev=2):
        """one nonlinear step on device arrays (of four levels)"""
        def dev():
            p = ctypes.c_void_p()
            assert self.stub.s.hipMalloc(ctypes.byref(p), ctypes.c_size_t(16 * 4 * self.lm_max)) == 0
            return p.value
        if not hasattr(self, "arrays"):
            self.arrays = (ctypes.c_void_p * 11)(*[dev() for _ in range(11)]), \
                (ctypes.c_void_p * 10)(*[dev() for _ in range(10)])
        r = (ctypes.c_double * nlev)(*[1.0] * nlev)
        lc = (ctypes.c_int * nlev)(*[self.l_max] * nlev)
        return self.L.mhx_nl_step(self.h, nlev, self.arrays[0], ctypes.c_size_t(self.lm_max), self.arrays[1], r, r, r,
                                  ctypes.c_double(1.0), lc, None)


def launched(entry, kernel):
    return entry[0] == "launch" and kernel in entry[1]


def check_filled(log, kernel, ptrs):
    """the tables at ptrs are allocated, and since then written whole by one
    launch of `kernel` and waited for"""
    for p in ptrs:
        assert p != "0", "null table"
        state = "none"
        for e in log:
            if e[0] == "malloc" and e[1] == p:
                state = "raw"
            elif e[0] == "free" and e[1] == p:
                state = "none"
            elif launched(e, kernel) and p in e[2:] and state != "none":
                state = "written"
            elif e[0] == "sync" and state == "written":
                state = "filled"
        assert state == "filled", (kernel, p, state)


def failed_first_call(st, precision, name):
    """Every way in which a call's resources can fail, then the same call
    again: it reads whole tables or reports an error, and nothing is lost."""
    p = st.plan(precision)
    assert p.call(name) == 0
    live = st.s.stub_live()
    p.close()
    failures = 0
    for n in range(1, 200):
        p = st.plan(precision)
        st.s.stub_fail(n)
        rc = p.call(name)
        st.s.stub_fail(0)
        if rc == 0:
            p.close()
            break
        failures += 1
        assert st.L.mhx_last_error()
        before = len(st.log())
        assert p.call(name) == 0, st.L.mhx_last_error()
        log = st.log()
        if name == "scal_to_spat":
            last = [e for e in log if launched(e, "k_p_tables")][-1]
            check_filled(log, "k_p_tables", last[4:6])
            check_filled(log, "k_crec64", [e for e in log if launched(e, "k_crec64")][-1][2:])
        elif name != "tables":
            check_filled(log, "k_plm_tables", [e for e in log if launched(e, "k_axi")][-1][2:])
        else:  # the export's own tables: allocated, written, copied and freed in the call
            again = log[before:]
            pair = [e for e in again if launched(e, "k_plm_tables")][0][2:4]
            assert [e[1] for e in again if e[0] == "malloc"] == pair
            assert sorted(e[1] for e in again if e[0] == "free") == sorted(pair)
        assert st.s.stub_live() == live, (n, st.s.stub_live(), live)
        p.close()
        assert st.s.stub_live() == 0
        st.s.stub_clear()
    assert failures > 0


def tables_at_creation(st, precision):
    """After its creation a plan's calls allocate, build and wait for nothing
    beyond their own work, and the table export leaves nothing behind."""
    p = st.plan(precision)
    for name in ("axi_to_spat", "toraxi_to_spat", "scal_to_spat", "spat_to_qst"):
        st.s.stub_clear()
        assert p.call(name) == 0, st.L.mhx_last_error()
        log = st.log()
        assert not [e for e in log if e[0] in ("malloc", "free", "memset", "sync")], (name, log)
        assert not [e for e in log if launched(e, "tables")], (name, log)
    live = st.s.stub_live()
    assert p.call("tables") == 0 and st.s.stub_live() == live
    p.close()


def analysis_pair_given_up(st):
    """The 2 pi w P, dP pair, from which the split tables are made, is not held
    besides the P-only tables: they take its memory, large enough for either."""
    for shape in (PLANS[SPLIT16], (17, 1, 28, 64), (31, 3, 40, 96)):
        st.s.stub_clear()
        p = st.plan(SPLIT16, shape=shape)
        log = st.log()
        pair = [e for e in log if launched(e, "k_plm_tables")][0][4:6]
        fill = [i for i, e in enumerate(log) if launched(e, "k_p_tables")][0]
        assert pair == log[fill][4:6]
        split = [i for i, e in enumerate(log) if launched(e, "k_split")]
        assert ["sync"] in log[split[-1]:fill]  # the split tables' kernels have read it
        for t in pair:
            size = [int(e[2]) for e in log if e[0] == "malloc" and e[1] == t][-1]
            assert [int(e[2]) for e in log[:fill] if e[0] == "memset" and e[1] == t][-1] <= size
        p.close()


def lds_per_device(st):
    """A kernel's LDS attribute is set on every device that launches it, once
    and for a larger size again."""
    def attributes(device, shape, precision, name):
        st.s.stub_device(device)
        p = st.plan(precision, shape=shape)
        st.s.stub_clear()
        for _ in range(2):
            assert (p.step() if name == "step" else p.call(name)) == 0, st.L.mhx_last_error()
        got = [(int(e[1]), e[2], int(e[3])) for e in st.log() if e[0] == "attribute"]
        p.close()
        return got
    # l_max, minc, n_theta, n_phi whose grid stage or epilogue takes over 64 KB
    for shape, precision, name in (((20, 1, 32, 1536), FP64, "step"), ((20, 1, 32, 1024), FP64, "step"),
                                   ((20, 1, 32, 3072), FP64, "step"), ((20, 1, 32, 768), SPLIT16, "step"),
                                   ((20, 1, 32, 3072), SPLIT16, "step"), ((240, 16, 32, 64), FP64, "spat_to_qst"),
                                   ((282, 16, 32, 64), FP64, "spat_to_qst")):
        first = attributes(0, shape, precision, name)
        assert first and all(d == 0 and n > 65536 for d, _, n in first), (shape, first)
        assert attributes(0, shape, precision, name) == []
        assert attributes(1, shape, precision, name) == [(1, k, n) for _, k, n in first], shape


def graph_destroyed_first(st, precision):
    """A plan's captured step goes before the streams and events it was
    captured on and the memory it addresses."""
    p = st.plan(precision)
    for _ in range(3):
        assert p.step() == 0, st.L.mhx_last_error()
    st.s.stub_clear()
    p.close()
    log = [e for e in st.log() if e[0] in ("destroy", "free")]
    assert log[0] == ["destroy", "exec"], log[:3]
    assert log.count(["destroy", "exec"]) == 1


def failed_growth(st, precision):
    """A step on more levels than the plan has room for, each of its
    allocations failing in turn, then a step on the plan's own number of
    levels: it finds every workspace it needs."""
    for n in range(1, 200):
        p = st.plan(precision, levels=2)
        assert p.step(2) == 0, st.L.mhx_last_error()
        st.s.stub_fail(n)
        rc = p.step(4)
        st.s.stub_fail(0)
        if rc == 0:
            break
        assert p.step(2) == 0, (n, st.L.mhx_last_error())
        st.s.stub_clear()
        assert p.step(2) == 0 and p.step(2) == 0
        assert "0" not in [e[1] for e in st.log() if e[0] == "memcpy"], n
        p.close()
    assert n > 6


def failed_rloop(st):
    """Every way in which a first radial loop's resources can fail, then the
    same call again: the theta factors it reads were copied to the device."""
    for n in range(1, 300):
        p = st.plan(FP64)
        p._L = p.L
        z = np.zeros((2, p.lm_max), dtype=np.complex128)
        rad = dict({k: np.ones(2) for k in sht.RLOOP_RAD}, **{k: np.full(2, 5, dtype=np.int32) for k in sht.RLOOP_RAD_INT})
        fields = {k: z for k in sht.RLOOP_IN}
        outs = {k: z.copy() for k in sht.RLOOP_OUT}
        phys = dict(l_conv=1, l_conv_nl=1, l_heat=1, l_heat_nl=1, l_mag=1, l_mag_LF=1, l_mag_nl=1)

        def call():
            sht.rloop(p, phys, 2, rad, fields, outs, np.zeros(2), np.zeros(2))
        st.s.stub_fail(n)
        try:
            call()
            break
        except sht.MhxError:
            st.s.stub_fail(0)
        call()
        size = str(5 * p.nt * 8)
        log = st.log()
        made = [i for i, e in enumerate(log) if e[0] == "malloc" and e[2] == size][-1]
        assert ["memcpy", log[made][1], size] in log[made:], n
        p.close()
        assert st.s.stub_live() == 0, n
        st.s.stub_clear()
    assert n > 10


if __name__ == "__main__":
    fn = globals()[sys.argv[3]]
    fn(Stub(sys.argv[1], sys.argv[2]), *[int(x) if x.isdigit() else x for x in sys.argv[4:]])
