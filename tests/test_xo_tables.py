"""The xoshiro skip tables hold the digits of every offset that a run can
reach: the longest run is the one whose accumulators fill the GPU's memory."""
import os
import re

import trois_photons as tp
from conftest import PKG

HBM, ACC, EVENTS = 288 * 10**9, 104, 10_000


def test_tables_reach_the_longest_run():
    text = open(os.path.join(PKG, "csrc", "tp_kernels.h")).read()
    digits = {k: int(re.search(rf"XO_{k}_DIGITS = (\d+)", text).group(1)) for k in "MB"}
    batches = HBM // ACC
    # faster-evgen draws 16.64 values an event on average and its stream is expanded in pieces of 172 032
    draws = 17 * EVENTS * batches + 2 * 172_032
    assert tp.BATCH_SIZE == EVENTS
    assert 16 ** digits["M"] > draws
    assert 16 ** digits["B"] > batches
    # the tables are made from that many of the 64 powers M^(2^k)
    assert 4 * digits["M"] <= 64
