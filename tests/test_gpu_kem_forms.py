"""The one-launch KEM kernels' forms by batch size: eight instances per workgroup,
then two or four groups of 32 (the other edges of the lane-pair forms and the
other sets: test_gpu_kem_pairs.py).

The bytes are compared with the VALU backend's chains of kernels, which share
neither the product kernels nor the workgroup layout, and a sample with the
CPU oracle.
"""
import numpy as np
import pytest

import oracle as O
import tmvp_amd as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with T.Context(0) as c:
        yield c


# Eight instances per workgroup (512, 513), then lane pairs with 48, 49 and 64
# (a second group), one full round, four groups (65: three used), four full
# groups, a second round.
SIZES = (512, 513, 1536, 1537, 2048, 2049, 4097, 8193, 16384, 16385, 32768, 32769)


@pytest.mark.parametrize("ps", ["lightsaber", "saber", "firesaber", "sable2"])
@pytest.mark.parametrize("batch", SIZES)
def test_forms_equal_chain(ctx, ps, batch):
    rng = np.random.default_rng(batch)
    seeds = rng.integers(0, 256, (batch, 96), dtype=np.uint8)
    pk, sk = T.run_kem_keypair(ctx, seeds, ps, T.MFMA)
    pk2, sk2 = T.run_kem_keypair(ctx, seeds, ps, T.VALU)
    assert np.array_equal(pk, pk2) and np.array_equal(sk, sk2)
    rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
    ct, ss = T.run_kem_encaps(ctx, pk, rnd, ps, T.MFMA)
    ct2, ss2 = T.run_kem_encaps(ctx, pk, rnd, ps, T.VALU)
    assert np.array_equal(ct, ct2) and np.array_equal(ss, ss2)
    bad = np.arange(batch % 5, batch, 5)
    ct[bad, rng.integers(0, ct.shape[1], bad.size)] ^= (1 << rng.integers(0, 8, bad.size)).astype(np.uint8)
    dec, fail = T.run_kem_decaps(ctx, ct, sk, ps, T.MFMA)
    dec2, fail2 = T.run_kem_decaps(ctx, ct, sk, ps, T.VALU)
    assert np.array_equal(dec, dec2) and np.array_equal(fail, fail2)
    assert np.array_equal(np.flatnonzero(fail), bad)
    sample = np.unique(np.r_[0, batch - 1, rng.integers(0, batch, 6)])
    want_pk, want_sk = O.kem_keypair_batch(ps, seeds[sample], nthreads=8)
    assert np.array_equal(pk[sample], want_pk) and np.array_equal(sk[sample], want_sk)
    assert np.array_equal(dec[sample], O.kem_dec_batch(ps, ct[sample], sk[sample], nthreads=8))


@pytest.mark.parametrize("batch", [1, 40, 16385])
def test_decaps_reports_out_of_range_secret(ctx, batch):
    """A Saber secret key whose coefficient 5 is 200, outside the matrix
    cores' int8 range, is reported; the same key repaired is not."""
    rng = np.random.default_rng(3)
    pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), "saber", T.MFMA)
    ct, _ = T.run_kem_encaps(ctx, pk, rng.integers(0, 256, (batch, 32), dtype=np.uint8), "saber", T.MFMA)
    bits = np.unpackbits(sk[-1], bitorder="little")
    kept = bits.copy()
    bits[5 * 13:6 * 13] = [(200 >> i) & 1 for i in range(13)]
    sk[-1] = np.packbits(bits, bitorder="little")
    with pytest.raises(T.TmvpError) as e:
        T.run_kem_decaps(ctx, ct, sk, "saber", T.MFMA)
    assert e.value.code == T.ERANGE
    sk[-1] = np.packbits(kept, bitorder="little")
    T.run_kem_decaps(ctx, ct, sk, "saber", T.MFMA)
