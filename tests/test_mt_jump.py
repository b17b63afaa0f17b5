"""The polynomials with which large dropout and bernoulli draws jump ahead in MT19937-64's words (host/kd_mt_jump.cpp),
against the generator itself, and what the first call pays for them."""
import ctypes
import subprocess
import sys

import numpy as np

import kd
import support

P = support.ptr
SYMBOL = "_ZN2kd19mt_jump_polynomialsEi"
BLOCKS, CHAINS, N = 64, 64, 312


def twist(old):
    new, first = np.empty_like(old), np.concatenate([old[1:], old[:1]])
    def mixed(a, b, far):
        y = (a & np.uint64(0xFFFFFFFF80000000)) | (b & np.uint64(0x7FFFFFFF))
        return far ^ (y >> np.uint64(1)) ^ np.where(y & np.uint64(1), np.uint64(0xB5026F5AA96619E9), np.uint64(0))
    new[:156] = mixed(old[:156], first[:156], old[156:])
    new[156:311] = mixed(old[156:311], first[156:311], new[:155])
    new[311:] = mixed(old[311:], new[:1], new[155:156])
    return new


def test_polynomials_reach_each_chain():
    lib = ctypes.CDLL(str(kd.LIB_PATH))
    state = np.zeros(N + 1, np.uint64)
    lib.kd_mt19937_64_seed(P(state), ctypes.c_uint64(99))
    words = [state[:N]]
    for _ in range(BLOCKS * (CHAINS - 1)):
        words.append(twist(words[-1]))
    words = np.concatenate(words)
    get = getattr(lib, SYMBOL)
    get.restype = ctypes.POINTER(ctypes.c_uint64)
    for count in (1, 2, 5, CHAINS - 1):  # asked for little by little
        table = np.ctypeslib.as_array(get(count), ((CHAINS - 1) * N,)).reshape(CHAINS - 1, N)
        bits = np.unpackbits(table[count - 1].view(np.uint8), bitorder="little")
        got = np.zeros(N, np.uint64)
        for k in np.flatnonzero(bits):
            got ^= words[k + 1:k + 1 + N]
        np.testing.assert_array_equal(got, words[N * BLOCKS * count:][:N])


def test_the_first_large_draw_waits_little_for_them():
    """All of them take 2.6 ms of a new process; a search for the recurrence in the generator's output took 41."""
    code = ("import ctypes, sys, time; lib = ctypes.CDLL(sys.argv[1]); t = time.process_time(); "
            "getattr(lib, sys.argv[2])(%d); print(time.process_time() - t)" % (CHAINS - 1))
    times = [float(subprocess.run([sys.executable, "-c", code, str(kd.LIB_PATH), SYMBOL], check=True, capture_output=True,
                                  text=True).stdout) for _ in range(3)]
    assert min(times) < 0.012, times
