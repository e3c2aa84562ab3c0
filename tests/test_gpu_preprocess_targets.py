"""Preprocess-stage read-start counts (no_pos_hash_pr) where a block of the coverage scan (4,096 columns)
adds up one target's counts in LDS and the others' directly: targets shorter than a thread's 16 columns,
targets that end inside a block, and one of several blocks, against the oracle bit for bit."""
import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [[30, 41, 4096, 35], [9000, 33, 4095], [37] * 300, [4097], [12300, 64, 64]])
def test_starts_per_target(lengths):
    print("[gpu] preprocess read starts over targets of", lengths[:4], flush=True)
    rng = np.random.default_rng(len(lengths) + lengths[0])
    refs = [("t%03d" % i, "".join(rng.choice(list("ACGT"), n))) for i, n in enumerate(lengths)]
    reads = []
    for t, n in enumerate(lengths):
        for pos in sorted(int(x) for x in rng.integers(0, max(1, n - 24), max(4, n // 6))):
            reads.append(dict(tid=t, pos=pos, cigar="24M", seq=refs[t][1][pos:pos + 24],
                              flag=16 if rng.random() < 0.5 else 0, x1=2 if rng.random() < 0.03 else 1))
    s = BuiltSample(Built(refs, reads))
    kw = dict(preprocess_stage=True, do_errors=False)
    args = B.api.make_error_count_args(s, **kw)
    hists, _, _, texts = O.error_count(args)
    res = B.api.error_count(s, **kw)
    assert np.array_equal(res.histograms[0], hists[0])
    assert np.array_equal(res.no_pos_hash_pr, texts["no_pos_hash_pr"], equal_nan=True)
