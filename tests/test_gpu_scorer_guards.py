"""The guards of the exact scorer: which candidates are decided by sums in any order (level 0), by a full fit
and close comparisons in read order (1) and wholly in read order (2).  Raising the guards sends candidates
from level 0 to the others, through the hand-over of single bisection steps among them, and must not change a
byte; nor must columns so deep, or tolerances so small, that the rounding of a sum passes the least
guards.  Every text is compared with the unscreened run's, which sums in read order, and the oracle's."""
import numpy as np
import pytest

import breseq_amd as B
import oracle_lib as O
from aln_builder import Built, BuiltSample
from parity_util import compare_gd
from test_gpu_scorer_levels import gd_text, sample

pytestmark = pytest.mark.gpu


def args_of(s, tol=None):
    ea = B.api.make_error_count_args(s, quality_max=42)
    _, _, l_o, texts = O.error_count(ea)
    table = O.read_log10_prob_table(texts["error_rates"], len(l_o))
    args = B.api.make_identify_args(s, table, ea.read_set_max, 42, [1.0], mode=B.POLYMORPHISM)
    args.polymorphism_precision_places = 8
    args.polymorphism_cutoff = 0.5
    if tol is not None:
        args.polymorphism_precision_decimal = tol
    return args


@pytest.mark.parametrize("depth,n_mapq", [(60, 1), (256, 1), (120, 40), (700, 40)])
def test_every_level(depth, n_mapq):
    print("[gpu] scorer guards: depth", depth, "MAPQs", n_mapq, flush=True)
    s = sample(depth + n_mapq, depth, list(range(42, 42 - n_mapq, -1)), n_sites=20)
    args = args_of(s)
    sess = B.Session().load(s)
    try:
        want = gd_text(sess, args, True)
        seen = [0, 0, 0]
        for guards in [(1e-8, 2e-12), (1e-2, 2e-12), (0.3, 2e-12), (1e-8, 1e-4), (1e-2, 1e-4), (1e9, 2e-12)]:
            sess.set_scorer_guards(*guards)
            assert gd_text(sess, args, False) == want, guards
            levels = sess.scorer_levels()
            print("[gpu]   guards", guards, "levels", levels, flush=True)
            assert sum(levels) == sess.timing()["candidates"]
            seen = [a + b for a, b in zip(seen, levels)]
            if guards == (1e-8, 2e-12):
                assert levels[0] > 0
            if guards == (1e9, 2e-12):
                assert levels[2] >= want.count("RA\t")
        assert min(seen) > 0
    finally:
        sess.close()
    compare_gd(want, O.identify_mutations(args)[0])


@pytest.mark.parametrize("tol", [1e-4, 1e-9, 1e-11, 1e-13])
def test_tolerances(tol):
    """A loop that ends a pass earlier or later changes a frequency by up to the tolerance."""
    print("[gpu] scorer guards: tolerance", tol, flush=True)
    s = sample(17, 300, [42], n_sites=40)
    args = args_of(s, tol)
    sess = B.Session().load(s)
    try:
        a, b = gd_text(sess, args, False), gd_text(sess, args, True)
    finally:
        sess.close()
    assert a == b and a.count("RA\t") > 10
    compare_gd(a, O.identify_mutations(args)[0])


def test_twenty_thousand_reads():
    print("[gpu] scorer guards: 20,000 reads a column", flush=True)
    rng = np.random.default_rng(8)
    ref = "".join(rng.choice(list("ACGT"), 100))
    alts = {30: 0.2, 41: 0.5, 44: 0.31, 52: 0.97}
    seqs = rng.choice(list("ACGT"), (20000, 40))
    keep = rng.random((20000, 40)) < 0.999
    base = np.array(list(ref[20:60]))
    seqs = np.where(keep, base, seqs)
    for p, f in alts.items():
        seqs[rng.random(20000) < f, p - 20] = "ACGT"[("ACGT".index(ref[p]) + 1) % 4]
    qual = rng.integers(20, 42, (20000, 40))
    reads = [dict(pos=20, cigar="40M", seq="".join(seqs[i]), qual=qual[i].tolist(), flag=16 * int(i % 3 == 0))
             for i in range(20000)]
    s = BuiltSample(Built([("t0", ref)], reads))
    args = args_of(s)
    sess = B.Session().load(s)
    try:
        a, levels = gd_text(sess, args, False), sess.scorer_levels()
        b = gd_text(sess, args, True)
    finally:
        sess.close()
    print("[gpu]   levels", levels, flush=True)
    assert a == b and a.count("RA\t") >= len(alts)
    compare_gd(a, O.identify_mutations(args)[0])
