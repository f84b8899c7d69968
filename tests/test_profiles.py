"""The committed profiles are of the committed kernels.

Each summary under profiles/ names the digest of the reader source it was taken
from; `bench.py` uses a summary only where that is the current source's. A
change to the kernels makes this fail until the profiles are taken again.
"""

import glob
import os

import pytest

import bench


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(bench.PROFILES, "*.txt"))),
                         ids=os.path.basename)
def test_profile_is_of_the_current_source(path):
    with open(path) as f:
        digests = [line.split(":")[1].strip() for line in f if line.startswith("source_sha256_16:")]
    assert digests == [bench.source_digest()]


def test_headline_traffic_is_reported():
    traffic = bench.measured_traffic("group_exact_kernel", "c2", 64, 16)
    assert traffic is not None and traffic["read_bytes"] > traffic["write_bytes"] > 0
