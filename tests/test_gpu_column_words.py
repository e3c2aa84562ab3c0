"""The column pass's word-wise loops (eight alignments at a time, eight columns to a lane) at their edges,
against the oracle: aligned spans of 1 to 200 columns at every offset to the 64-column windows, trims at
either end, N bases, low qualities, alignments left over from the groups of eight, and reads that the
loops do not take (qualities of N bases past the maximum, qualities above 127); with a window shared by
its block's wavefronts (few windows) and a wavefront per window (many), and quality cutoffs from none to
all; with likelihood tables of up to the most that is staged in LDS (7 MAPQs of 43 qualities) and beyond."""
import re

import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from parity_util import compare_gd

pytestmark = pytest.mark.gpu

FEW, MANY = 1500, 64 * 4200


def sample(seed, length, n, q=(2, 42), n_mapq=1, odd=False, deep=None):
    rng = np.random.default_rng(seed)
    ref = "".join(rng.choice(list("ACGT"), length))
    ref = ref[:700] + "N" + ref[701:]
    sites = {int(p): str(rng.choice([c for c in "ACGT" if c != ref[p]])) for p in rng.integers(80, 1400, 14)}
    reads = []
    for i in range(n):
        m = int(rng.choice([1, 7, 8, 9, 40, 63, 64, 65, 100, 200]))
        if deep is not None:
            pos = deep
        elif length > FEW and i % 4 == 0:
            pos = int(rng.integers(0, length - m))
        else:
            pos = int(rng.integers(0, FEW - m))
        seq = [sites[x] if x in sites and rng.random() < 0.6 else ref[x] for x in range(pos, pos + m)]
        qual = rng.integers(q[0], q[1] + 1, m)
        for k in np.nonzero(rng.random(m) < 0.02)[0]:
            seq[k] = str(rng.choice(list("ACGTN")))
            if odd and seq[k] == "N":
                qual[k] = 250
        xl, xr = (int(rng.integers(0, 6)), int(rng.integers(0, 6))) if rng.random() < 0.7 else (-1, -1)
        reads.append(dict(pos=pos, cigar="%dM" % m, seq="".join(seq), qual=[int(x) for x in qual], xl=xl, xr=xr,
                          flag=16 if rng.random() < 0.5 else 0, mapq=42 - int(rng.integers(0, n_mapq)),
                          x1=2 if rng.random() < 0.02 else 1))
    reads.sort(key=lambda r: r["pos"])
    return BuiltSample(Built([("t0", ref)], reads))


def check(s, q_max, **kw):
    args = B.api.make_error_count_args(s, quality_max=q_max)
    _, _, l_o, texts = O.error_count(args)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    iargs = B.api.make_identify_args(s, table, args.read_set_max, q_max, [2.0], mode=B.POLYMORPHISM, **kw)
    gd_o, _ = O.identify_mutations(iargs)
    gd_g = B.api.identify_mutations(s, table, args.read_set_max, q_max, [2.0], mode=B.POLYMORPHISM, **kw)
    if q_max > 128:   # the scorer's quality histogram, for the KS test of strand and quality bias, ends at 127
        gd_o, gd_g = (re.sub(r"\t(ks_quality|bias_)\w*=[^\t\n]*", "", x) for x in (gd_o, gd_g))
    n, same, errs = compare_gd(gd_g, gd_o)
    print("[gpu]   entries", n, "identical", same, errs, flush=True)
    return n


@pytest.mark.parametrize("length", [FEW, MANY])
@pytest.mark.parametrize("n,n_mapq", [(60, 1), (900, 1), (900, 7), (900, 8), (900, 40)])
def test_spans_and_trims(length, n, n_mapq):
    print("[gpu] column words: length", length, "reads", n, "MAPQs", n_mapq, flush=True)
    assert check(sample(n + length, length, n, n_mapq=n_mapq), 43) > 3


@pytest.mark.parametrize("length", [FEW, MANY])
def test_deep_column(length):
    """More alignments of one start than the byte-wise counts hold steps of."""
    print("[gpu] column words: deep, length", length, flush=True)
    assert check(sample(3, length, 2600, deep=200), 43) > 0


@pytest.mark.parametrize("q,q_max,odd", [((2, 42), 43, True), ((100, 199), 200, False), ((60, 127), 128, False),
                                         ((60, 128), 129, False)])
def test_reads_outside_the_word_loops(q, q_max, odd):
    print("[gpu] column words: qualities", q, q_max, odd, flush=True)
    assert check(sample(11, FEW, 700, q=q, odd=odd), q_max) > 3


@pytest.mark.parametrize("cutoff", [0, 2, 20, 42, 43, 127, 200])
def test_quality_cutoffs(cutoff):
    print("[gpu] column words: cutoff", cutoff, flush=True)
    check(sample(12, FEW, 500), 43, base_quality_cutoff=cutoff)
