"""The host entry points' staging rings (four pieces of 512 KB each way):
operands that end on either side of a piece, of the ring and of several rings,
against the device entry points; what is left in page-locked memory afterwards;
and how much of it is held."""
import numpy as np
import pytest

import tmvp_amd as T
from test_gpu_host_secrets import memory_type, page_locked_copies

pytestmark = pytest.mark.gpu


@pytest.fixture()
def lib():
    lib = T.load_library()
    yield lib
    assert lib.tmvp_host_release() == 0


def page_locked_bytes(locked):
    n = 0
    for line in open("/proc/self/maps").read().splitlines():
        parts = line.split(maxsplit=5)
        lo, hi = (int(x, 16) for x in parts[0].split("-"))
        if len(parts) == 6 and parts[5].startswith("/dev/dri/") and memory_type(lo) == locked:
            n += hi - lo
    return n


# LightSaber: 704 bytes in and 768 out per encapsulation, 2304 in per
# decapsulation: one piece, the ring and two rings lie at these and one more.
@pytest.mark.parametrize("batch", [682, 683, 744, 745, 910, 911, 2730, 2731, 2978, 2979, 5957, 5958, 7281, 7282, 20000])
def test_staged_calls_equal_device_calls(lib, batch):
    rng = np.random.default_rng(batch)
    at = lambda x: x.ctypes.data
    with T.Context(0) as ctx:
        pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), "lightsaber")
        rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
        want_ct, want_ss = T.run_kem_encaps(ctx, pk, rnd, "lightsaber")
    mark = T.pinned_array((64,))
    mark[:32] = rng.integers(0, 256, 32, dtype=np.uint8)
    locked = memory_type(at(mark))
    held = page_locked_bytes(locked)
    assert lib.tmvp_host_configure(0, batch, T.LIGHTSABER, 1, T.SABLE2) == 0
    last = batch - 1
    patterns = [x.tobytes() for x in (mark[:32], rnd[0], rnd[last], want_ss[0], want_ss[last], sk[0, :32], sk[0, -32:],
                                      sk[last // 2, :32], sk[last, :32], sk[last, -32:])]
    for _ in range(2):
        ct, ss, dec = np.zeros_like(want_ct), np.zeros_like(want_ss), np.zeros_like(want_ss)
        assert lib.tmvp_host_set_randomness(at(rnd), batch) == 0
        lib.saber_enc(0, at(ss), at(pk), at(ct))
        assert lib.tmvp_host_status() == 0
        assert np.array_equal(ct, want_ct) and np.array_equal(ss, want_ss)
        assert page_locked_copies(patterns, locked) == [1] + 9 * [0]
        lib.saber_dec(0, at(ct), at(pk), at(sk), at(dec))
        assert lib.tmvp_host_status() == 0
        assert np.array_equal(dec, want_ss)
        assert page_locked_copies(patterns, locked) == [1] + 9 * [0]
    assert page_locked_bytes(locked) - held <= 2 * (2 << 20) + 2 * 8192
