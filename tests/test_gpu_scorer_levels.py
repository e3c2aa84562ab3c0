"""The exact scorer's two ways to a result: EM loops with sums in any order over the distinct table keys,
with every decision and printed digit checked against a guard, and the reference's sums in read order
(every candidate of an unscreened run).  Both must print the same genome diff, and the oracle's, on
candidates at the edges of the kernel: a read or two, 15-17 and 255-257 reads (the ordered chain's
groups), columns of more distinct keys than the scorer keeps rows for, tables of many MAPQs (too large to
count keys directly, and past the candidate test's histogram), and more printed digits than the
unordered sums can vouch for."""
import ctypes as C

import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from breseq_amd import _lib as L
from parity_util import compare_gd

pytestmark = pytest.mark.gpu


def sample(seed, depth, mapqs, n_sites=12, length=400, read_length=40, freq=(0.05, 1.0)):
    rng = np.random.default_rng(seed)
    ref = "".join(rng.choice(list("ACGT"), length))
    sites = {int(p): (str(rng.choice([c for c in "ACGT" if c != ref[p]])), float(rng.uniform(*freq)))
             for p in rng.choice(np.arange(60, length - 60), n_sites, replace=False)}
    n = max(1, int(round(depth * (length - read_length) / read_length)))
    reads = []
    for pos in sorted(int(x) for x in rng.integers(0, length - read_length + 1, n)):
        seq = list(ref[pos:pos + read_length])
        qual = [int(q) for q in np.clip(rng.normal(30, 7, read_length).round(), 2, 41)]
        for i in range(read_length):
            s = sites.get(pos + i)
            if s and rng.random() < s[1]:
                seq[i] = s[0]
            if rng.random() < 10 ** (-qual[i] / 10):
                seq[i] = str(rng.choice(list("ACGT")))
        reads.append(dict(pos=pos, cigar="%dM" % read_length, seq="".join(seq), qual=qual,
                          flag=16 if rng.random() < 0.5 else 0, mapq=int(rng.choice(mapqs))))
    return BuiltSample(Built([("t0", ref)], reads))


def gd_text(sess, args, unscreened):
    lib, res, st = L.lib(), C.c_void_p(), L.Status()
    fn = lib.bsq_session_identify_unscreened if unscreened else lib.bsq_session_identify
    L.check(fn(sess._h, C.byref(args), C.byref(res), C.byref(st)), st)
    return B.api._im_texts(res)[0]


@pytest.mark.parametrize("depth,n_mapq,places,mode", [
    (1.5, 1, 8, B.POLYMORPHISM), (16, 1, 8, B.POLYMORPHISM), (16, 1, 3, B.CONSENSUS), (60, 1, 8, B.POLYMORPHISM),
    (256, 1, 8, B.POLYMORPHISM), (60, 40, 8, B.POLYMORPHISM), (700, 40, 8, B.POLYMORPHISM), (40, 1, 14, B.POLYMORPHISM),
    (2500, 3, 8, B.POLYMORPHISM)])
def test_both_ways_print_the_same(depth, n_mapq, places, mode):
    print("[gpu] scorer levels: depth", depth, "MAPQs", n_mapq, "places", places, mode, flush=True)
    s = sample(int(depth) + 100 * n_mapq + places, depth, list(range(42, 42 - n_mapq, -1)))
    ea = B.api.make_error_count_args(s, quality_max=42)
    _, _, l_o, texts = O.error_count(ea)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    args = B.api.make_identify_args(s, table, ea.read_set_max, 42, [1.0], mode=mode)
    args.polymorphism_precision_places = places
    args.polymorphism_cutoff = 0.5   # candidates of every kind, weak ones among them
    sess = B.Session().load(s)
    try:
        a, b = gd_text(sess, args, False), gd_text(sess, args, True)
    finally:
        sess.close()
    assert a == b
    n, same, errs = compare_gd(a, O.identify_mutations(args)[0])
    print("[gpu]   entries", n, "identical", same, errs, flush=True)
    assert ("RA\t" in a) == (depth > 2)
