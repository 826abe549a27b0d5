"""fci_sigma_device_noalloc (sigma whose scratch is the library's static device array) against
fci_sigma_device (scratch the solver allocates), through the C ABI, on two calls in a row, the
second with a smaller problem, in FP64 and in FP32; and the size limit."""
import ctypes
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

_d = ctypes.POINTER(ctypes.c_double)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _lib():
    import forte_amd
    L = ctypes.CDLL(forte_amd.LIBRARY_PATH)
    L.fci_create.argtypes = [ctypes.c_int] * 3 + [_d] * 5 + [ctypes.c_double, ctypes.POINTER(ctypes.c_void_p)]
    L.fci_destroy.argtypes = [ctypes.c_void_p]
    L.fci_last_error.restype = ctypes.c_char_p
    L.fci_last_error.argtypes = [ctypes.c_void_p]
    L.fci_ndet.restype = ctypes.c_int64
    L.fci_ndet.argtypes = [ctypes.c_void_p]
    for f in ("fci_sigma_device", "fci_sigma_device_noalloc"):
        getattr(L, f).argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
    L.fci_device_alloc.argtypes = [ctypes.c_size_t, ctypes.POINTER(ctypes.c_void_p)]
    L.fci_device_free.argtypes = [ctypes.c_void_p]
    L.fci_device_upload.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    L.fci_device_download.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    return L


def _create(L, n, na, nb, seed):
    from oracle import oracle as O
    h, eri = O.seeded_integrals(n, seed)
    aa, ab = O.chem_to_forte(eri)
    keep = [np.ascontiguousarray(x) for x in (h, h, aa, ab, aa)]
    hnd = ctypes.c_void_p()
    rc = L.fci_create(n, na, nb, *[x.ctypes.data_as(_d) for x in keep], 0.21, ctypes.byref(hnd))
    assert rc == 0, L.fci_last_error(None)
    return hnd


class Dev:
    def __init__(self, L, nbytes):
        self.L, self.p = L, ctypes.c_void_p()
        assert L.fci_device_alloc(nbytes, ctypes.byref(self.p)) == 0

    def __del__(self):
        self.L.fci_device_free(self.p)


def _sigma_pair(L, hnd, C, dtype):
    nb = C.nbytes
    c, s1, s2 = Dev(L, nb), Dev(L, nb), Dev(L, nb)
    assert L.fci_device_upload(c.p, C.ctypes.data, nb) == 0
    # fill the no-alloc output with garbage first: the entry point must overwrite every element
    junk = np.full_like(C, 7.0)
    assert L.fci_device_upload(s2.p, junk.ctypes.data, nb) == 0
    assert L.fci_sigma_device(hnd, c.p, s1.p, dtype, None) == 0, L.fci_last_error(hnd)
    rc = L.fci_sigma_device_noalloc(hnd, c.p, s2.p, dtype, None)
    assert rc == 0, L.fci_last_error(hnd)
    a, b = np.empty_like(C), np.empty_like(C)
    assert L.fci_device_download(a.ctypes.data, s1.p, nb) == 0
    assert L.fci_device_download(b.ctypes.data, s2.p, nb) == 0
    return a, b


@pytest.mark.parametrize("dtype", [0, 1])
def test_noalloc_sigma_matches_allocating_sigma(dtype):
    L = _lib()
    # two calls in a row on the shared scratch: CAS(12,12) (853,776 determinants), then a smaller
    # problem with unequal spins
    for (n, na, nb, seed) in [(12, 6, 6, 3), (9, 4, 3, 5)]:
        say(f"noalloc sigma dtype {dtype} n={n} na={na} nb={nb}")
        hnd = _create(L, n, na, nb, seed)
        nd = L.fci_ndet(hnd)
        x = np.random.default_rng(seed).standard_normal(nd)
        x /= np.linalg.norm(x)
        C = x if dtype == 0 else x.astype(np.float32)
        ref, got = _sigma_pair(L, hnd, C, dtype)
        err = np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max()
        say(f"  max |noalloc - allocating| / max|sigma| = {err:.2e}")
        # FP64: the alpha-beta row sums add in scheduling order (last-bit differences);
        # FP32: rounded from those FP64 row sums
        assert err < (1e-13 if dtype == 0 else 1e-6)
        L.fci_destroy(hnd)


@pytest.mark.parametrize("n,na,nb", [(13, 6, 2), (12, 2, 6)])
def test_noalloc_sigma_other_routes(n, na, nb):
    """FP64 above 924 strings, whose clique intermediates live in the scratch, and a dense one with long beta rows;
    bounds as above."""
    L = _lib()
    say(f"noalloc sigma n={n} na={na} nb={nb}")
    hnd = _create(L, n, na, nb, 4)
    C = np.random.default_rng(4).standard_normal(L.fci_ndet(hnd))
    ref, got = _sigma_pair(L, hnd, C, 0)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-13
    L.fci_destroy(hnd)


def test_noalloc_refuses_problems_beyond_the_scratch():
    L = _lib()
    say("noalloc size limit: CAS(14,14)")
    hnd = _create(L, 14, 7, 7, 2)
    nd = L.fci_ndet(hnd)
    c, s = Dev(L, nd * 4), Dev(L, nd * 4)
    rc = L.fci_sigma_device_noalloc(hnd, c.p, s.p, 1, None)
    assert rc == -1
    assert b"scratch" in L.fci_last_error(hnd)
    assert L.fci_sigma_device_noalloc(hnd, c.p, s.p, 3, None) == -1
    L.fci_destroy(hnd)
