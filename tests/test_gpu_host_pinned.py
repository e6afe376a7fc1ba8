"""The host entry points on page-locked caller buffers: read and written in
place, mixed with pageable ones, off the 16-byte grid, past the staging's limit,
against the device entry points; and no slower than from pageable memory."""
import time

import numpy as np
import pytest

import tmvp_amd as T

pytestmark = pytest.mark.gpu


@pytest.fixture()
def lib():
    lib = T.load_library()
    yield lib
    assert lib.tmvp_host_release() == 0


def held(data, kind):
    """A copy of data in pageable ("p") or page-locked memory, "l" on the
    16-byte grid and "o" eight bytes off it."""
    if kind == "p":
        return data.copy()
    off = 8 if kind == "o" else 0
    out = T.pinned_array((data.size + off,))[off:].reshape(data.shape)
    out[...] = data
    return out


def configure(lib, ps, batch):
    sable = ps.startswith("sable")
    pid = T.PARAM_SET_NAMES[ps]
    assert lib.tmvp_host_configure(0, 1 if sable else batch, T.SABER if sable else pid, batch if sable else 1,
                                   pid if sable else T.SABLE2) == 0
    return sable


def at(x):
    return x.ctypes.data


def enc(lib, sable, ss, pk, ct):
    lib.SABLE_enc(at(ss), at(pk), at(ct), 0) if sable else lib.saber_enc(0, at(ss), at(pk), at(ct))
    assert lib.tmvp_host_status() == 0


def dec(lib, sable, ct, pk, sk, ss):
    lib.SABLE_dec(at(ct), at(pk), at(sk), at(ss), 0) if sable else lib.saber_dec(0, at(ct), at(pk), at(sk), at(ss))
    assert lib.tmvp_host_status() == 0


# kinds of pk, ct, ss of an encapsulation and of ct, sk, ss of a decapsulation
@pytest.mark.parametrize("kinds", ["lll", "lpp", "plp", "ppl", "llp", "pll", "ooo", "lol"])
@pytest.mark.parametrize("ps,batch", [("saber", 3), ("sable2", 700), ("sable1", 4100)])
def test_page_locked_buffers_equal_device_calls(lib, ps, batch, kinds):
    check(lib, ps, batch, kinds)


@pytest.mark.parametrize("kinds", ["lll", "plp", "ppp"])
def test_past_the_staging_limit(lib, kinds):
    check(lib, "firesaber", 13000, kinds)


def check(lib, ps, batch, kinds):
    rng = np.random.default_rng(batch)
    with T.Context(0) as ctx:
        pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), ps)
        rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
        want_ct, want_ss = T.run_kem_encaps(ctx, pk, rnd, ps)
    sable = configure(lib, ps, batch)
    h_pk, ct, ss = held(pk, kinds[0]), held(np.zeros_like(want_ct), kinds[1]), held(np.zeros_like(want_ss), kinds[2])
    assert lib.tmvp_host_set_randomness(at(rnd), batch) == 0
    enc(lib, sable, ss, h_pk, ct)
    assert np.array_equal(ct, want_ct) and np.array_equal(ss, want_ss) and np.array_equal(h_pk, pk)
    h_ct, h_sk, out = held(want_ct, kinds[0]), held(sk, kinds[1]), held(np.zeros_like(want_ss), kinds[2])
    dec(lib, sable, h_ct, h_pk, h_sk, out)
    assert np.array_equal(out, want_ss) and np.array_equal(h_ct, want_ct) and np.array_equal(h_sk, sk)


def test_page_locked_buffers_pay_no_host_copies(lib):
    """8192 Saber encapsulations: 8 MB in and 9 MB out, whose copies on the host
    take about 0.3 of the call from pageable memory."""
    ps, batch = "saber", 8192
    p = T.get_params(ps)
    sable = configure(lib, ps, batch)
    rng = np.random.default_rng(1)
    best = {}
    for kind in "pl":
        pk = held(rng.integers(0, 256, (batch, p["pk_bytes"]), dtype=np.uint8), kind)
        ct, ss = held(np.zeros((batch, p["ct_bytes"]), np.uint8), kind), held(np.zeros((batch, 32), np.uint8), kind)
        rnd = np.zeros((batch, 32), np.uint8)
        times = []
        for _ in range(25):
            assert lib.tmvp_host_set_randomness(at(rnd), batch) == 0
            t = time.perf_counter()
            enc(lib, sable, ss, pk, ct)
            times.append(time.perf_counter() - t)
        best[kind] = min(times)
    assert best["l"] < 0.9 * best["p"], best
