"""The one-launch KEM's lane-pair kernels where their last workgroup or group
of 32 is nearly empty or full, and Sable types 1 and 3 in each of their forms:
bytes against the VALU backend's chains and the CPU oracle, as in
test_gpu_kem_forms.py.

Workgroups hold ceil(B / 32) instances up to 2048, 64 up to 16384 (two groups of
32), beyond that at most 128 (four groups): tmvp_kem_form.h.
"""
import numpy as np
import pytest

import tmvp_amd as T
from test_gpu_kem_forms import test_forms_equal_chain as equal_chain_and_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with T.Context(0) as c:
        yield c


# Rows of lanes up to 768.  Two groups: 25 a workgroup (the second empty), 33 (one
# instance in it), 49; of 64, the last workgroup holds 1, 31, 32, 33 or 63.
EDGES = (767, 768, 769, 1025, 1537, 2049, 2079, 2080, 2081, 2111)
# Four groups: 65 a workgroup (one instance in the third group; the last workgroup
# holds 5 in one), 97 (one in the fourth), full, 65 in two rounds.
FOUR = (16384, 16385, 24832, 32768, 32769)


@pytest.mark.parametrize("ps", ["lightsaber", "saber", "firesaber", "sable1", "sable2", "sable3"])
@pytest.mark.parametrize("batch", EDGES)
def test_rows_and_two_groups_edges(ctx, ps, batch):
    equal_chain_and_oracle(ctx, ps, batch)


@pytest.mark.parametrize("ps", ["sable1", "sable3"])
@pytest.mark.parametrize("batch", FOUR)
def test_full_and_four_groups(ctx, ps, batch):
    equal_chain_and_oracle(ctx, ps, batch)


@pytest.mark.parametrize("ps", ["lightsaber", "saber", "firesaber", "sable2"])
def test_four_groups_single_instance(ctx, ps):
    equal_chain_and_oracle(ctx, ps, 24832)


@pytest.mark.parametrize("batch", [1000, 2049, 16384])
def test_two_groups_report_out_of_range_secret(ctx, batch):
    """The last instance's coefficient 5 is 200, outside the matrix cores'
    int8 range: reported; the same key repaired is not."""
    rng = np.random.default_rng(batch)
    pk, sk = T.run_kem_keypair(ctx, rng.integers(0, 256, (batch, 96), dtype=np.uint8), "saber")
    ct, _ = T.run_kem_encaps(ctx, pk, rng.integers(0, 256, (batch, 32), dtype=np.uint8), "saber")
    kept = sk[-1].copy()
    bits = np.unpackbits(kept, bitorder="little")
    bits[5 * 13:6 * 13] = [(200 >> i) & 1 for i in range(13)]
    sk[-1] = np.packbits(bits, bitorder="little")
    with pytest.raises(T.TmvpError) as e:
        T.run_kem_decaps(ctx, ct, sk, "saber")
    assert e.value.code == T.ERANGE
    sk[-1] = kept
    T.run_kem_decaps(ctx, ct, sk, "saber")
