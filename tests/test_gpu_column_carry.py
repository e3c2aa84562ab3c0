"""The column pass reads an alignment's qualities in groups of eight bytes, which hold the end of the packed
alignment before it where it begins inside a group.  Qualities of 255 there (a redundant alignment's, an
N base's) must not reach its own first base: the FP32 sums of every column stay within the bound of a
summation of the FP64 ones, with a window shared by its block's wavefronts and a wavefront per window,
and with the likelihood table staged in LDS and read from memory."""
import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from parity_util import compare_gd

pytestmark = pytest.mark.gpu

FEW, MANY = 1500, 64 * 4200
Q = 43


def sample(length, n_mapq, top):
    """Pairs in file order: an alignment of 8k bases whose last quality is 255, then a unique one that begins
    at every offset to a group of eight columns."""
    rng = np.random.default_rng(length + n_mapq)
    ref = "".join(rng.choice(list("ACGT"), length))
    reads = []
    for i in range(400):
        pos = 100 + 3 * i + int(rng.integers(0, 3))
        m = 8 * int(rng.integers(1, 8))
        seq, qual = ref[pos:pos + m], [30] * (m - 1) + [255]
        if i % 2:   # unique, of an N base at the end
            seq = seq[:-1] + "N"
        reads.append(dict(pos=pos, cigar="%dM" % m, seq=seq, qual=qual, x1=1 if i % 2 else 2, flag=16 * int(rng.integers(0, 2))))
        m = int(rng.integers(9, 60))
        reads.append(dict(pos=pos, cigar="%dM" % m, seq=ref[pos:pos + m], qual=[int(x) for x in rng.integers(2, top + 1, m)],
                          x1=1, flag=16 * int(rng.integers(0, 2)), mapq=42 - int(rng.integers(0, n_mapq))))
    return BuiltSample(Built([("t0", ref)], reads))


@pytest.mark.parametrize("length", [FEW, MANY])
@pytest.mark.parametrize("n_mapq,top", [(1, Q - 3), (1, Q - 1), (40, Q - 1)])
def test_quality_of_the_alignment_before(length, n_mapq, top):
    print("[gpu] column carry: length", length, "MAPQs", n_mapq, "qualities to", top, flush=True)
    s = sample(length, n_mapq, top)
    args = B.api.make_error_count_args(s, quality_max=Q)
    _, _, l_o, texts = O.error_count(args)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    sess = B.Session().load(s)
    try:
        rep = sess.precision_audit(table, args.read_set_max, Q, [2.0], mode=B.POLYMORPHISM)
    finally:
        sess.close()
    print("[gpu]  ", rep, flush=True)
    assert rep["columns"] > 1000
    assert rep["decision_mismatches"] == 0 and rep["count_mismatches"] == 0
    # at most 60 alignments a column: their terms rounded once each, then the additions
    assert rep["max_rel_error"] < 62 * 2.0 ** -24
    iargs = B.api.make_identify_args(s, table, args.read_set_max, Q, [2.0], mode=B.POLYMORPHISM)
    compare_gd(B.api.identify_mutations(s, table, args.read_set_max, Q, [2.0], mode=B.POLYMORPHISM),
               O.identify_mutations(iargs)[0])
