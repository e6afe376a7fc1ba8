"""The one-launch KEM kernels' small-batch form (a state on a row of lanes,
eight instances per workgroup in two groups of four; 1535 instances run on
lane pairs, 48 to a workgroup).

Every set at the group and workgroup edges, against the VALU backend's chains,
which share neither the permutation nor the product kernels, and the CPU
oracle.
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


@pytest.mark.parametrize("ps", ["lightsaber", "saber", "firesaber", "sable1", "sable2", "sable3"])
@pytest.mark.parametrize("batch", [1, 3, 4, 5, 8, 9, 1535])
def test_small_batches_equal_chain_and_oracle(ctx, ps, batch):
    rng = np.random.default_rng(batch)
    seeds = rng.integers(0, 256, (batch, 96), dtype=np.uint8)
    pk, sk = T.run_kem_keypair(ctx, seeds, ps, T.MFMA)
    pk2, sk2 = T.run_kem_keypair(ctx, seeds, ps, T.VALU)
    assert np.array_equal(pk, pk2) and np.array_equal(sk, sk2)
    rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
    ct, ss = T.run_kem_encaps(ctx, pk, rnd, ps, T.MFMA)
    ct2, ss2 = T.run_kem_encaps(ctx, pk, rnd, ps, T.VALU)
    assert np.array_equal(ct, ct2) and np.array_equal(ss, ss2)
    bad = np.arange(batch % 3, batch, 3)
    ct[bad, rng.integers(0, ct.shape[1], bad.size)] ^= (1 << rng.integers(0, 8, bad.size)).astype(np.uint8)
    dec, fail = T.run_kem_decaps(ctx, ct, sk, ps, T.MFMA)
    dec2, fail2 = T.run_kem_decaps(ctx, ct, sk, ps, T.VALU)
    assert np.array_equal(dec, dec2) and np.array_equal(fail, fail2)
    assert np.array_equal(np.flatnonzero(fail), bad)
    sample = np.unique(np.r_[0, batch - 1, rng.integers(0, batch, 9)])
    want_pk, want_sk = O.kem_keypair_batch(ps, seeds[sample], nthreads=8)
    assert np.array_equal(pk[sample], want_pk) and np.array_equal(sk[sample], want_sk)
    assert np.array_equal(dec[sample], O.kem_dec_batch(ps, ct[sample], sk[sample], nthreads=8))
