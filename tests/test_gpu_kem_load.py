"""The chains' sponge kernels with more waves than SIMDs (the permutation's
waves in step): keyed batches on either side of the line, against the plain
calls.  The plain chains cross their lines in test_gpu_kem_forms.py and
test_gpu_kem_pairs.py (16384, 16385, 32768, 32769)."""
import numpy as np
import pytest

import tmvp_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ps", ["lightsaber", "saber", "sable3"])
@pytest.mark.parametrize("op,batch", [(T.SRV_ENCAPS, 32768), (T.SRV_ENCAPS, 32769), (T.SRV_DECAPS, 16384),
                                      (T.SRV_DECAPS, 16385), (T.SRV_DECAPS, 32769)])
def test_keyed_batches_equal_plain_calls(ps, op, batch):
    rng = np.random.default_rng(batch)
    keys = rng.integers(0, 64, batch).astype(np.int32)
    rnd = rng.integers(0, 256, (batch, 32), dtype=np.uint8)
    with T.Context(0) as ctx:
        pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (64, 96), dtype=np.uint8), ps)
        ct, ss = T.run_kem_encaps(ctx, pk[keys], rnd, ps)
        if op == T.SRV_DECAPS:
            bad = np.arange(0, batch, 7)
            ct[bad, 3] ^= 4
            ss, fail = T.run_kem_decaps(ctx, ct, sk[keys], ps)
            assert np.array_equal(np.flatnonzero(fail), bad)
        srv = T.Server(ctx, max_batch=batch, slots=1)
        try:
            first = srv.add_keys(ps, pk, sk)
            _, out = srv.submit(op, ps, keys + first, rnd if op == T.SRV_ENCAPS else ct)
            done = []
            while not done:
                done = srv.poll(timeout_us=100000)
            assert done[0]["status"] == T.OK and done[0]["batch_instances"] == batch
            for got, want in zip(out, (ct, ss) if op == T.SRV_ENCAPS else (ss, fail)):
                assert np.array_equal(got, want)
        finally:
            srv.close()
