"""Checks on the library built for the CPU, each run by tests/test_emu.py in a process of its
own: checks.py NAME (TONTO_GPU_LIB names the library, the address sanitizer is preloaded)."""
import ctypes
import dataclasses
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))

import numpy as np  # noqa: E402

import oracle.oracle as oracle  # noqa: E402
from tonto_amd.basis import Molecule  # noqa: E402
from tonto_amd.geometry import water_cluster  # noqa: E402
from tonto_amd.gpu import JKEngine, TGPUError, lib  # noqa: E402


class Emu:
    """The stand-in's log and switches."""

    def __init__(self):
        self.L = lib()
        self.L.emu_entry.restype = ctypes.c_char_p
        self.L.emu_stream.restype = ctypes.c_void_p

    def log(self):
        out = []
        v = (ctypes.c_longlong * 6)()
        for i in range(self.L.emu_size()):
            name = self.L.emu_entry(i, v).decode()
            out.append((name,) + tuple(v))
        return out

    def fail(self, name, n):
        self.L.emu_fail(name.encode(), n)

    def launches(self):
        """(kernel, stream, threads, grid x, grid y, block, LDS bytes) of every launch"""
        return [e for e in self.log() if e[5] > 0]


def _ints(v):
    return (ctypes.c_int * len(v))(*v)


def launch_limits():
    """Bin pairs of a class pair that together exceed one launch's 2^32 threads go into several,
    none of them dropped; what one bin pair alone exceeds is refused."""
    e = Emu()
    e.L.emu_execute(0)

    def launch(n_bra, n_ket, variant, mixed=0):
        e.L.emu_clear()
        rc = e.L.emu_launch_1000(len(n_bra), _ints(n_bra), _ints(n_ket), variant, mixed)
        return rc, e.launches()
    for mixed in (0, 1):
        # one work-group per bra pair (long ket segments), four bra pairs per work-group, both
        for n_bra, n_ket, groups in (([9000000] * 4, [300] * 4, 36000000), ([60000000] * 3, [9] * 3, 45000000),
                                     ([9000000, 9000001, 16000000], [300, 9, 300], 25000000 + 2250001)):
            rc, ls = launch(n_bra, n_ket, 0, mixed)
            assert rc == 0
            assert all(threads < 2 ** 32 for _, _, threads, *_ in ls), ls
            assert sum(l[3] for l in ls) == groups, ls
        # wavefront form
        rc, ls = launch([40000000] * 3, [9] * 3, 1, mixed)
        assert rc == 0
        assert all(threads < 2 ** 32 for _, _, threads, *_ in ls), ls
        assert sum(l[3] for l in ls) == 120000000 * (1 + mixed), ls
    # an ordinary class pair stays one launch
    rc, ls = launch([1000] * 16, [9] * 16, 0)
    assert rc == 0 and len(ls) == 1 and ls[0][3] == 4000
    # too large by itself; more parts than a launch holds
    assert launch([20000000], [300], 0)[0] != 0
    assert launch([70000000], [9], 1)[0] != 0
    assert launch([1] * 17, [9] * 17, 0)[0] != 0
    # Schwarz: 16 lanes per pair
    e.L.emu_clear()
    n = (1 << 28) + 5
    e.L.emu_schwarz_10(3, n)
    ls = e.launches()
    assert all(threads < 2 ** 32 for _, _, threads, *_ in ls), ls
    assert sum(4 * l[3] for l in ls) >= n


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return 0.5 * A @ A.T / n


class Build:
    """A context with its matrices (device memory is host memory here)."""

    def __init__(self, mol, seed=0, **options):
        self.mol, self.eng = mol, JKEngine(mol, **options)
        self.max_I = self.eng.schwarz()
        self.P = _density(self.eng.n_bf, seed)
        self.J, self.K = np.empty_like(self.P), np.empty_like(self.P)

    def run(self, **flags):
        self.J.fill(np.nan)
        self.K.fill(np.nan)
        self.eng.make_r_JK_device(self.P.ctypes.data, self.J.ctypes.data, self.K.ctypes.data, **flags)
        return self.J.copy(), self.K.copy()


def failing_runtime_calls():
    """A fork, join, launch or capture that fails ends the build with an error, forked streams are
    joined all the same, and the next build is right."""
    e = Emu()
    b = Build(water_cluster(1, "STO-3G", seed=1))
    J0, K0 = b.run()

    def fails(name, n, what, **flags):
        e.L.emu_clear()
        e.fail(name, n)
        try:
            b.run(**flags)
        except TGPUError:
            pass
        else:
            raise AssertionError(f"{what} failed and the build went on")
        finally:
            e.fail("", -1)
        failed = e.log()
        b.eng.set_cutoffs_scaled(1.0)  # (a captured build runs at its capture only)
        J, K = b.run(**flags)
        assert abs(J - J0).max() < 1e-14 and abs(K - K0).max() < 1e-14, what
        return failed
    for flags in (dict(), dict(graph=True)):
        if flags:
            b.eng.set_cutoffs_scaled(1.0)  # (drops the captured build)
        e.L.emu_clear()
        b.run(**flags)
        log = e.log()
        waited = {x[2] for x in log if x[0] == "hipStreamWaitEvent"}
        records = [x for x in log if x[0] == "hipEventRecord"]
        n_fork = len([x for x in log if x[0] == "hipStreamWaitEvent"])
        n_launch = len(e.launches())
        assert n_fork >= 6 and len(records) >= 4 and n_launch > 6, (n_fork, records, n_launch)
        for n, r in enumerate(records):
            if r[2] in waited and n in (0, 1, 2, len(records) - 1, len(records) - 2):  # (the others are timing events)
                b.eng.set_cutoffs_scaled(1.0)
                fails("hipEventRecord", n, f"record {n} of {flags}", **flags)
        for n in sorted({0, 1, 2, n_fork // 2, n_fork - 1}):
            b.eng.set_cutoffs_scaled(1.0)
            log = fails("hipStreamWaitEvent", n, f"wait {n} of {flags}", **flags)
            # no launch on a side stream without a join or a host wait after it, unless captured
            if not flags:
                done = {x[1] for x in log if x[0] in ("hipEventRecord", "hipStreamSynchronize")}
                assert {l[1] for l in log if l[5] > 0} <= done | {0}, log
        for n in (0, 8, n_launch - 1):
            b.eng.set_cutoffs_scaled(1.0)
            fails("launch", n, f"launch {n} of {flags}", **flags)
    # a failed capture: its side streams go, and no later build uses them
    b.eng.set_cutoffs_scaled(1.0)
    log = fails("hipStreamEndCapture", 0, "the capture", graph=True)
    gone = {x[1] for x in log if x[0] == "hipStreamDestroy"}
    assert len(gone) == 3, log
    assert gone.isdisjoint({l[1] for l in e.launches()[len(log):]})
    # no side streams to be had: the build runs in series
    e.fail("hipStreamCreate", 0)
    b2 = Build(water_cluster(1, "STO-3G", seed=1))
    e.fail("", -1)
    J, K = b2.run()
    assert abs(J - J0).max() < 1e-14 and abs(K - K0).max() < 1e-14


def kept_workspace():
    """A destroyed context leaves its workspace to the next; an allocation that fails frees it and
    is tried again."""
    e = Emu()
    mol = water_cluster(1, "cc-pVTZ", seed=1)
    first = JKEngine(mol)
    first.schwarz()
    first.close()
    e.L.emu_clear()
    second = JKEngine(mol)
    second.schwarz()
    with_kept = len([x for x in e.log() if x[0] == "hipMalloc"])
    third = JKEngine(mol)
    e.L.emu_clear()
    third.schwarz()
    alone = len([x for x in e.log() if x[0] == "hipMalloc"])
    second.close()  # (leaves the larger workspace or the same)
    e.L.emu_clear()
    fourth = JKEngine(mol)
    n_create = len([x for x in e.log() if x[0] == "hipMalloc"])
    fourth.schwarz()
    assert with_kept - n_create == alone - 1, (with_kept, n_create, alone)
    fourth.close()
    e.fail("hipMalloc", 0)
    fifth = JKEngine(mol)  # the kept buffer makes room
    e.fail("hipMalloc", 0)
    try:
        JKEngine(mol)  # nothing is kept now
    except TGPUError:
        pass
    else:
        raise AssertionError("no error")
    e.fail("", -1)
    e.L.emu_clear_error()
    fifth.schwarz()
    third.close()
    fifth.close()


def side_streams_per_stream():
    """Builds on two streams share no side stream, builds on one stream share theirs; with more
    streams than sets the longest unused set goes round."""
    e = Emu()
    mol = water_cluster(1, "STO-3G", seed=1)
    streams = [e.L.emu_stream() for _ in range(11)]
    b = [Build(mol), Build(mol)]
    J0, K0 = b[0].run()

    def side(k, s):
        b[k].eng.set_stream(s)
        e.L.emu_clear()
        J, K = b[k].run()
        assert abs(J - J0).max() < 1e-14 and abs(K - K0).max() < 1e-14
        return frozenset(x[1] for x in e.launches()) - {own(s)}

    def own(s):
        return ctypes.cast(s, ctypes.POINTER(ctypes.c_int))[0]
    first = side(0, streams[0])
    assert len(first) == 3
    assert not first & side(1, streams[1])
    assert side(1, streams[0]) == first == side(0, streams[0])
    e.L.emu_execute(0)
    J0 = K0 = np.full_like(J0, np.nan)
    sets = []
    for s in streams:
        b[0].eng.set_stream(s)
        e.L.emu_clear()
        b[0].run()
        sets.append(frozenset(x[1] for x in e.launches()) - {own(s)})
    assert all(len(x) == 3 for x in sets) and len(set(sets)) == 8, sets


def captured_by_the_caller():
    """A build on a stream that the caller captures makes no stream or event and forks nothing."""
    e = Emu()
    b = Build(water_cluster(1, "STO-3G", seed=1))
    J0, K0 = b.run()
    s = e.L.emu_stream()
    ctypes.cast(s, ctypes.POINTER(ctypes.c_int))[1] = 1  # (its capture flag)
    b.eng.set_stream(s)
    e.L.emu_clear()
    J, K = b.run()
    assert abs(J - J0).max() < 1e-14 and abs(K - K0).max() < 1e-14
    log = e.log()
    assert not [x for x in log if "Create" in x[0] or x[0] in ("hipMalloc", "hipStreamWaitEvent")], log
    assert len({x[1] for x in e.launches()}) == 1


def _spd_system():
    """Four atoms far enough apart that quartets over all four lose primitive pairs, some all of
    them; contracted and single primitives; 12 shells."""
    m = Molecule.from_angstrom(["O"] * 4, [[0, 0, 0], [2.7, 0.4, -0.3], [0.9, 5.6, 0.5], [6.1, 1.0, 4.2]], "6-31G(d)")
    shells, bf = [], 0
    for s in m.shells:
        n = len(s.exps)
        if n > (3 if s.atom == 0 else 1) or (s.atom == 0 and n == 1 and s.l < 2):
            continue
        shells.append(dataclasses.replace(s, first_bf=bf))
        bf += s.n_comp
    m.shells, m.n_bf = shells, bf
    return m


def _f_system():
    """Three atoms with an f, a d, a p and an s shell (cc-pVTZ), the first s contracted."""
    m = Molecule.from_angstrom(["O"] * 4, [[0, 0, 0], [2.7, 0.4, -0.3], [0.9, 5.6, 0.5], [6.1, 1.0, 4.2]], "cc-pVTZ")
    shells, bf, seen = [], 0, set()
    for s in m.shells:
        if (s.atom, s.l) in seen or (s.l < 2 and len(s.exps) > 1 and (s.atom or s.l)) or (s.atom == 3 and s.l > 1):
            continue
        seen.add((s.atom, s.l))
        shells.append(dataclasses.replace(s, first_bf=bf))
        bf += s.n_comp
    m.shells, m.n_bf = shells, bf
    return m


def _compare(eng, mol, P, cut, mixed, tol):
    J, K = eng.make_r_JK(P, mixed=mixed)
    Jo, Ko, so = oracle.OracleSystem(mol).make_r_JK(P, schwarz=cut, max_I=eng.schwarz(), return_stats=True)
    st = eng.stats()
    print("max|dJ| %.1e max|dK| %.1e, %d quartets" % (abs(J - Jo).max(), abs(K - Ko).max(), st["quartets"]), flush=True)
    assert st["quartets"] == so["quartets"] and st["prim_quartets"] == so["prim_quartets"]
    assert max(abs(J - Jo).max(), abs(K - Ko).max()) <= tol
    return st


def wavefront_forms():
    """Every class pair up to d shells in the wavefront form (FP64, FP32 and both in a build; the
    last team of a chunk without a quartet, primitive lists that are empty, several passes over
    rows and columns) and the lane form, against the oracle; the Schwarz table in both bases."""
    mol = _spd_system()
    o = oracle.OracleSystem(mol)
    P = _density(mol.n_bf, 5)
    for thr, tol in ((1e-9, 1e-11), (1e30, 2e-5), (1e-3, 2e-5)):
        e = JKEngine(mol, schwarz=1e-13, fp32_threshold=thr)
        assert abs(e.schwarz() - o.schwarz()).max() < 1e-13
        for k in range(21):
            e.set_variant(k, 1)
            e.set_ket_chunk(k, (16, 32, 64)[k % 3])
        st = _compare(e, mol, P, 1e-13, thr > 1e-9, tol)
        assert (st["fp32_quartets"] > 0) == (thr > 1e-9)
    assert st["fp32_quartets"] < st["quartets"]
    e = JKEngine(mol, schwarz=1e-13)
    _compare(e, mol, P, 1e-13, False, 1e-11)
    e = JKEngine(mol, spherical=True)
    assert abs(e.schwarz() - o.schwarz_sph()).max() < 1e-13


def f_shells():
    """Class pairs with f shells: both forms, the workspace as large as its launches need and as
    small as the allocation-free build may leave it, both bases."""
    mol = _f_system()
    o = oracle.OracleSystem(mol)
    P = _density(mol.n_bf, 5)
    for wave, thr, tol in ((1, 1e-9, 1e-11), (1, 1e-3, 2e-5), (0, 1e-9, 1e-11)):
        e = JKEngine(mol, schwarz=1e-12, fp32_threshold=thr)
        assert abs(e.schwarz() - o.schwarz()).max() < 1e-13
        for k in range(55):
            try:
                e.set_variant(k, wave)
            except TGPUError:  # only the wavefront form
                pass
            e.set_ket_chunk(k, (16, 32, 64)[k % 3])
        _compare(e, mol, P, 1e-12, thr > 1e-9, tol)
    Jo, Ko = o.make_r_JK(P, schwarz=1e-12, max_I=e.schwarz())
    J, K = np.zeros_like(P), np.zeros_like(P)
    e.make_r_JK_device_noalloc(P.ctypes.data, J.ctypes.data, K.ctypes.data)
    assert max(abs(J - Jo).max(), abs(K - Ko).max()) < 1e-11
    e = JKEngine(mol, spherical=True)
    assert abs(e.schwarz() - o.schwarz_sph()).max() < 1e-13


def lane_forms():
    """The lane form's kinds of K rows (one bra pair per work-group, a wavefront's own; all of
    them, some, none in LDS), a batch, J or K alone, UHF and the allocation-free build."""
    mol = _spd_system()
    P = _density(mol.n_bf, 6)
    for kets, budget in (("0", None), ("0", "15900"), ("1000000", None), ("1000000", "24000"), ("1000000", "15000")):
        os.environ["TGPU_KROW_MIN_KETS"] = kets
        if budget:
            os.environ["TGPU_KROW_BUDGET"] = budget
        e = JKEngine(mol, schwarz=1e-13)
        os.environ.pop("TGPU_KROW_BUDGET", None)
        _compare(e, mol, P, 1e-13, False, 1e-11)
    del os.environ["TGPU_KROW_MIN_KETS"]
    max_I = e.schwarz()
    o = oracle.OracleSystem(mol)
    Jo, Ko = o.make_r_JK(P, schwarz=1e-13, max_I=max_I)
    J, K = np.zeros_like(P), np.zeros_like(P)
    for only in ("J", "K", None):
        e.make_r_JK_device_noalloc(P.ctypes.data, J.ctypes.data, K.ctypes.data, only=only)
        assert only == "K" or abs(J - Jo).max() < 1e-11
        assert only == "J" or abs(K - Ko).max() < 1e-11
    P2 = _density(mol.n_bf, 7)
    for x, y in zip(e.make_u_JK(P, P2), o.make_u_JK(P, P2, schwarz=1e-13, max_I=max_I)):
        assert abs(x - y).max() < 1e-11
    mols = [water_cluster(1, "STO-3G", seed=1), mol, water_cluster(2, "STO-3G", seed=2)]
    Ps = [_density(m.n_bf, i) for i, m in enumerate(mols)]
    b = JKEngine(mols, schwarz=1e-12)
    max_I = b.schwarz()
    for i, (m, p, J, K) in enumerate(zip(mols, Ps, *b.make_r_JK(Ps))):
        Jo, Ko = oracle.OracleSystem(m).make_r_JK(p, schwarz=1e-12, max_I=max_I[b.pair_off[i]:b.pair_off[i + 1]])
        assert max(abs(J - Jo).max(), abs(K - Ko).max()) < 1e-11


if __name__ == "__main__":
    globals()[sys.argv[1]]()
    print("passed")
