"""The host entry points' staging keeps no secrets: after a call, the coins,
the secret key and the shared key are found in no page-locked memory of the
process."""
import ctypes

import numpy as np
import pytest

import tmvp_amd as T

pytestmark = pytest.mark.gpu


class Attributes(ctypes.Structure):
    """The head of hipPointerAttribute_t; the rest is room."""
    _fields_ = [("type", ctypes.c_int), ("device", ctypes.c_int), ("room", ctypes.c_uint8 * 248)]


def memory_type(address):
    a = Attributes()
    f = T.hip().hipPointerGetAttributes
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p]
    rc = f(ctypes.byref(a), address)
    T.hip().hipGetLastError()  # pageable memory may report an error: clear it
    return a.type if rc == 0 else None


def page_locked_copies(patterns, locked):
    """How often each pattern lies in page-locked memory, whose allocations are
    mappings of the GPU's device file."""
    found = [0] * len(patterns)
    for line in open("/proc/self/maps").read().splitlines():
        parts = line.split(maxsplit=5)
        lo, hi = (int(x, 16) for x in parts[0].split("-"))
        if len(parts) == 6 and parts[5].startswith("/dev/dri/") and parts[1].startswith("rw") and memory_type(lo) == locked:
            data = ctypes.string_at(lo, hi - lo)
            for k, want in enumerate(patterns):
                found[k] += data.count(want)
    return found


@pytest.mark.parametrize("ps,batch", [("saber", 3), ("sable2", 700), ("firesaber", 1200)])
def test_no_secret_stays_in_page_locked_memory(ps, batch):
    rng = np.random.default_rng(batch)
    lib = T.load_library()
    at = lambda x: x.ctypes.data
    sable, pid, p = ps.startswith("sable"), T.PARAM_SET_NAMES[ps], T.get_params(ps)
    with T.Context(0) as ctx:
        pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), ps)
    rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
    ct, ss, out = np.zeros((batch, p["ct_bytes"]), np.uint8), np.zeros((batch, 32), np.uint8), np.zeros((batch, 32), np.uint8)
    assert lib.tmvp_host_configure(0, 1 if sable else batch, T.SABER if sable else pid, batch if sable else 1,
                                   pid if sable else T.SABLE2) == 0
    # the search finds a pattern in page-locked memory
    control = T.pinned_array((64,))
    mark = rng.integers(0, 256, 32, dtype=np.uint8)
    control[:32] = mark
    locked = memory_type(at(control))
    assert memory_type(at(rnd)) != locked
    assert lib.tmvp_host_set_randomness(at(rnd), batch) == 0
    lib.SABLE_enc(at(ss), at(pk), at(ct), 0) if sable else lib.saber_enc(0, at(ss), at(pk), at(ct))
    assert lib.tmvp_host_status() == 0
    last = batch - 1
    secrets = [mark, rnd[0], rnd[last], ss[0], ss[last], sk[0, :32], sk[0, -32:], sk[last, :32], sk[last, -32:]]
    patterns = [x.tobytes() for x in secrets]
    assert page_locked_copies(patterns, locked) == [1] + 8 * [0]
    lib.SABLE_dec(at(ct), at(pk), at(sk), at(out), 0) if sable else lib.saber_dec(0, at(ct), at(pk), at(sk), at(out))
    assert lib.tmvp_host_status() == 0
    assert np.array_equal(out, ss)
    assert page_locked_copies(patterns, locked) == [1] + 8 * [0]
    assert lib.tmvp_host_release() == 0
