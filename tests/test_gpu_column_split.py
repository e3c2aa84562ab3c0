"""The column pass on either side of the line between a wavefront per window and windows shared by a block,
which follows from the most alignments of a window and those of them that go one at a time: no read, one to
four in one of 24 windows, and reads that cross a window's end, single runs and reads with a deletion, against the
oracle."""
import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from parity_util import compare_gd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 26])
@pytest.mark.parametrize("cigar", ["24M", "12M1D12M"])
def test_few_alignments_a_window(n, cigar):
    print("[gpu] column split:", n, "reads of", cigar, flush=True)
    rng = np.random.default_rng(n)
    ref = "".join(rng.choice(list("ACGT"), 24 * 64 - 1))
    reads = []
    for pos in sorted(int(x) for x in rng.integers(745, 766, n)):
        seq = list(ref[pos:pos + 12] + ref[pos + (13 if "D" in cigar else 12):])[:24]
        if pos <= 766 < pos + 12:
            seq[766 - pos] = "ACGT"[("ACGT".index(ref[766]) + 1) % 4]
        reads.append(dict(pos=pos, cigar=cigar, seq="".join(seq), flag=16 * int(rng.integers(0, 2))))
    s = BuiltSample(Built([("t0", ref)], reads))
    ea = B.api.make_error_count_args(s, quality_max=42)
    _, _, l_o, texts = O.error_count(ea)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    kw = dict(mode=B.POLYMORPHISM)
    args = B.api.make_identify_args(s, table, ea.read_set_max, 42, [2.0], **kw)
    compare_gd(B.api.identify_mutations(s, table, ea.read_set_max, 42, [2.0], **kw), O.identify_mutations(args)[0])
