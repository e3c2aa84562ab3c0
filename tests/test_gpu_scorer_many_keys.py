"""Candidate test and exact scorer on likelihood tables of any number of MAPQs: a column's distinct keys are found through
hashes (the candidate test's from the third MAPQ of one read file on, of 256 to 4,096 slots), and the
scorer's rows of them are in LDS at each of its three sizes, or read from the table (more distinct keys than
rows fit), with the read list in LDS and in device memory.  Screened and unscreened runs print the same
genome diff, and the oracle's."""
import pytest

import breseq_amd as B
import oracle_lib as O
from parity_util import compare_gd
from test_gpu_scorer_guards import args_of
from test_gpu_scorer_levels import gd_text, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,n_mapq", [(30, 5), (30, 6), (100, 40), (200, 10), (330, 40), (500, 20), (1200, 7), (1700, 10),
                                          (1700, 40), (3200, 40), (3200, 2)])
def test_many_mapqs(depth, n_mapq):
    print("[gpu] scorer keys: depth", depth, "MAPQs", n_mapq, flush=True)
    s = sample(depth + n_mapq, depth, list(range(42, 42 - n_mapq, -1)))
    args = args_of(s)
    sess = B.Session().load(s)
    try:
        a, levels = gd_text(sess, args, False), sess.scorer_levels()
        b = gd_text(sess, args, True)
    finally:
        sess.close()
    print("[gpu]   levels", levels, flush=True)
    assert a == b
    n, same, errs = compare_gd(a, O.identify_mutations(args)[0])
    print("[gpu]   entries", n, "identical", same, errs, flush=True)
    assert a.count("RA\t") >= 8
    # what the column pass's bound lets through of some 390 columns is tested again, whatever the table's size
    assert sum(levels) < 200
