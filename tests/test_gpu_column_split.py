"""The column pass on either side of the line between a wavefront per window and windows shared by a block:
24 windows with just fewer and just more aligned bases than windows in each, one read, and none, against
the oracle."""
import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from parity_util import compare_gd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 22, 23, 24, 25, 26])   # of 24 bases: 24 windows of 24 from 24 reads on
def test_few_bases_a_window(n):
    print("[gpu] column split:", n, "reads", flush=True)
    rng = np.random.default_rng(n)
    ref = "".join(rng.choice(list("ACGT"), 24 * 64 - 1))
    reads = []
    for pos in sorted(int(x) for x in rng.integers(700, 760, n)):
        seq = list(ref[pos:pos + 24])
        if pos <= 750 < pos + 24:
            seq[750 - pos] = "ACGT"[("ACGT".index(ref[750]) + 1) % 4]
        reads.append(dict(pos=pos, cigar="24M", seq="".join(seq), flag=16 * int(rng.integers(0, 2))))
    s = BuiltSample(Built([("t0", ref)], reads))
    ea = B.api.make_error_count_args(s, quality_max=42)
    _, _, l_o, texts = O.error_count(ea)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    kw = dict(mode=B.POLYMORPHISM)
    args = B.api.make_identify_args(s, table, ea.read_set_max, 42, [2.0], **kw)
    compare_gd(B.api.identify_mutations(s, table, ea.read_set_max, 42, [2.0], **kw), O.identify_mutations(args)[0])
