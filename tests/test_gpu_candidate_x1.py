"""The candidate test before the exact scorer counts the reads that the scorer does: those of X1 = 0 as well
as X1 = 1.  A variant that only X1 = 0 reads carry is found, by a screened and an unscreened run alike, as
the oracle finds it (single-run reads, and reads with a deletion)."""
import ctypes as C

import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from breseq_amd import _lib as L

pytestmark = pytest.mark.gpu


def texts(s, args):
    lib, out = L.lib(), []
    sess = B.Session().load(s)
    try:
        for fn in (lib.bsq_session_identify, lib.bsq_session_identify_unscreened):
            res, st = C.c_void_p(), L.Status()
            L.check(fn(sess._h, C.byref(args), C.byref(res), C.byref(st)), st)
            out.append(B.api._im_texts(res)[0])
    finally:
        sess.close()
    return out


def evidence(text):
    return [ln.split("\t")[3:] for ln in text.splitlines() if ln.startswith("RA\t")]


@pytest.mark.parametrize("cigar", ["40M", "10M1D30M"])
def test_variant_of_x1_zero_reads(cigar):
    print("[gpu] candidates: variant on X1 = 0 reads,", cigar, flush=True)
    rng = np.random.default_rng(4)
    ref = "".join(rng.choice(list("ACGT"), 300))
    at, alt = 150, "ACGT"[("ACGT".index(ref[150]) + 1) % 4]
    reads = []
    for i in range(240):
        pos = int(rng.integers(0, 255))
        zero = i % 4 == 0
        seq = list(ref[pos:pos + 10] + ref[pos + 11:pos + 41]) if zero and cigar != "40M" else list(ref[pos:pos + 40])
        k = at - pos - (1 if zero and cigar != "40M" and at - pos > 10 else 0)
        if zero and 0 <= k < 40 and at != pos + 10:
            seq[k] = alt
        reads.append(dict(pos=pos, cigar=cigar if zero else "40M", seq="".join(seq), qual=[int(x) for x in rng.integers(20, 40, 40)],
                          flag=16 * int(rng.integers(0, 2)), x1=0 if zero else 1))
    reads.sort(key=lambda r: r["pos"])
    s = BuiltSample(Built([("t0", ref)], reads))
    ea = B.api.make_error_count_args(s, quality_max=42)
    _, _, l_o, ec = O.error_count(ea)
    table = O.read_log10_prob_table(ec["error_rates"], len(l_o))
    args = B.api.make_identify_args(s, table, ea.read_set_max, 42, [1.0], mode=B.POLYMORPHISM)
    screened, unscreened = texts(s, args)
    assert screened == unscreened
    found = evidence(screened)
    assert [f[1] for f in found].count(str(at + 1)) == 1
    # (coverage sums of infinite 1/X1 are compared nowhere: RA entries only)
    assert [f[:5] for f in found] == [f[:5] for f in evidence(O.identify_mutations(args)[0])]
