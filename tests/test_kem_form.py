"""The one-launch KEM's form by batch size, for every size up to 70000.

The rule (csrc/tmvp_kem_form.h, plain C++) is compiled for the host.  A call has
to cover its batch with workgroups that hold their instances, and has to leave
room for the calls of seven other streams: up to one round of the two-group
form it takes no more CUs than workgroups of 64 need or an eighth of the chip,
and eight calls on rows of lanes (two workgroups to a CU) fit in one and a half
rounds.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "asfand-tmvp_amd", "csrc")
CUS, MOST = 256, 70000
PROGRAM = r"""
#include <stdio.h>
#include "tmvp_kem_form.h"
int main()
{
    for (int64_t b = 1; b <= %d; b++) {
        const tmvp::KemForm f = tmvp::kem_form(b);
        printf("%%d %%d %%lld\n", f.groups, f.per, (long long)f.blocks);
    }
}
"""


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("form")
    (d / "form.cpp").write_text(PROGRAM % MOST)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "form.cpp"), "-o", str(d / "form")], check=True)
    out = subprocess.run([str(d / "form")], check=True, capture_output=True, text=True).stdout
    got = np.array([line.split() for line in out.splitlines()], dtype=np.int64)
    assert got.shape == (MOST, 3)
    return got


def test_workgroups_cover_the_batch(forms):
    b = np.arange(1, MOST + 1)
    groups, per, blocks = forms.T
    assert set(np.unique(groups)) == {0, 2, 4}
    assert np.all(blocks * per >= b) and np.all((blocks - 1) * per < b)
    assert np.all(per <= np.where(groups == 0, 8, 32 * groups)) and np.all(per >= 1)


def test_calls_leave_room_for_other_streams(forms):
    b = np.arange(1, MOST + 1)
    groups, per, blocks = forms.T
    rows, two, four = groups == 0, groups == 2, groups == 4
    assert np.all(8 * blocks[rows] <= 3 * CUS)
    assert np.all(blocks[two] <= np.maximum(CUS // 8, -(-b[two] // 64)))
    assert np.all(b[four] > 64 * CUS) and np.all(blocks[four] <= CUS * -(-b[four] // (128 * CUS)))
