"""Checks on the library built for the CPU, each run by tests/test_emu.py in a process of its
own: checks.py NAME (TONTO_GPU_LIB names the library, the address sanitizer is preloaded)."""
import ctypes
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))

from tonto_amd.gpu import lib  # noqa: E402


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


if __name__ == "__main__":
    globals()[sys.argv[1]]()
    print("passed")
