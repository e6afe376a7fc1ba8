"""The host entry points' staging: batches on either side of a piece's end and
of the limit above which the runtime copies, against the device entry points."""
import numpy as np
import pytest

import tmvp_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ps", ["saber", "sable2"])
@pytest.mark.parametrize("batch", [1, 511, 512, 513, 585, 586, 16384, 16385])
def test_staged_calls_equal_device_calls(ps, batch):
    rng = np.random.default_rng(batch)
    lib, sable = T.load_library(), ps == "sable2"
    at = lambda x: x.ctypes.data
    with T.Context(0) as ctx:
        pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), ps)
        rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
        want_ct, want_ss = T.run_kem_encaps(ctx, pk, rnd, ps)
    assert lib.tmvp_host_configure(0, 1 if sable else batch, T.SABER, batch if sable else 1, T.SABLE2) == 0
    ct, ss, dec = np.zeros_like(want_ct), np.zeros_like(want_ss), np.zeros_like(want_ss)
    assert lib.tmvp_host_set_randomness(at(rnd), batch) == 0
    if sable:
        lib.SABLE_enc(at(ss), at(pk), at(ct), 0)
    else:
        lib.saber_enc(0, at(ss), at(pk), at(ct))
    assert lib.tmvp_host_status() == 0
    assert np.array_equal(ct, want_ct) and np.array_equal(ss, want_ss)
    if sable:
        lib.SABLE_dec(at(ct), at(pk), at(sk), at(dec), 0)
    else:
        lib.saber_dec(0, at(ct), at(pk), at(sk), at(dec))
    assert lib.tmvp_host_status() == 0
    assert np.array_equal(dec, want_ss)
