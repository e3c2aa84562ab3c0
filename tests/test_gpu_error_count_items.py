"""error_count where a wavefront's lanes share its alignments' runs in items of eight positions: runs of
one base up to beyond the longest that goes in one turn (8 * 40 positions), every alignment of the run
to the items, more and fewer runs than lanes, soft clips behind a hard clip (whose pairs reach past the
run), single-base indels, both strands, many alignments of one start, several read files up to the
largest count table, and bases and qualities that are refused; against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

import breseq_amd as B
from breseq_amd import _lib as L
import oracle_lib as O
from aln_builder import Built, BuiltSample

pytestmark = pytest.mark.gpu

CIGARS = ["{m}M", "{s}S{m}M", "{m}M{s}S", "{m}M{s}S3H", "2H{s}S{m}M", "{m}M1D{k}M", "{m}M1I{k}M", "{m}M{k}=2X",
          "{m}M3N{k}M"]


def sample(seed, lengths, n, files=1, one_start=False):
    rng = np.random.default_rng(seed)
    ref = "".join(rng.choice(list("ACGT"), 4000))
    ref = ref[:1500] + "NNN" + ref[1503:]
    reads = []
    for i in range(n):
        m, s, k = int(lengths[i % len(lengths)]), int(rng.integers(1, 12)), int(rng.integers(1, 9))
        cigar = CIGARS[i % len(CIGARS) if i % 3 else 0].format(m=m, s=s, k=k)
        pos = 700 if one_start else int(rng.integers(0, 4000 - m - 30))
        seq, x, num = [], pos, ""
        for c in cigar:
            if c.isdigit():
                num += c
                continue
            l, num = int(num), ""
            if c in "M=X":
                seq.append("".join(b if rng.random() > 0.05 else rng.choice(list("ACGTN")) for b in ref[x:x + l]))
            elif c in "IS":
                seq.append("".join(rng.choice(list("ACGTN"), l)))
            x += l if c in "M=XDN" else 0
        seq = "".join(seq)
        reads.append(dict(pos=pos, cigar=cigar, seq=seq, qual=rng.integers(2, 43, len(seq)).astype(np.uint8),
                          flag=16 if rng.random() < 0.5 else 0, x1=2 if rng.random() < 0.05 else 1,
                          rg=int(rng.integers(0, files)) if files > 1 else -1))
    reads.sort(key=lambda r: r["pos"])
    b = Built([("t0", ref)], reads)
    if files > 1:
        b.base = (C.c_uint32 * files)(*range(files))
        b.count = (C.c_uint32 * files)(*([1] * files))
        b.rf_names = (C.c_char_p * files)(*[b"reads%d" % i for i in range(files)])
        b.read_files = L.ReadFiles(files, b.base, b.count, files, b.rf_names)
    return BuiltSample(b)


def check(s, q_max=None):
    args = B.api.make_error_count_args(s, quality_max=q_max)
    hists, counts, _, _ = O.error_count(args)
    res = B.api.error_count(s, quality_max=q_max)
    assert np.array_equal(res.histograms[0], hists[0])
    assert np.array_equal(res.counts, counts.astype(np.uint64))
    assert res.counts.sum() > 0


@pytest.mark.parametrize("lengths,n", [([1, 2, 7, 8, 9, 15, 16, 17], 400), ([150], 65), ([36, 150], 64),
                                       ([300, 313, 314, 320, 321], 63), ([640, 1000, 2500, 5], 30), ([100], 1)])
def test_run_lengths(lengths, n):
    print("[gpu] error_count items, runs of", lengths, n, flush=True)
    check(sample(n, lengths, n))


@pytest.mark.parametrize("files", [3, 15])
def test_read_files(files):
    """15 read files of 43 qualities: the largest count table that is accepted."""
    print("[gpu] error_count items, read files", files, flush=True)
    check(sample(files, [40, 90], 500, files=files))


def test_one_start():
    print("[gpu] error_count items, one start", flush=True)
    check(sample(7, [50, 50, 50, 77], 700, one_start=True))


@pytest.mark.parametrize("what", [0, 3, 7, 9, 12, 14, 16, 31, 129, "quality", "reference"])
def test_refused(what):
    """A base code that is no base, a quality at the maximum, a reference letter that is neither a base
    nor N, each at one position of one alignment; a quality at the maximum of an N base is accepted."""
    print("[gpu] error_count items, refused", what, flush=True)
    for at in range(0, 24, 5):
        s = sample(5, [60], 100)
        b = s.b
        j = int(b.seq_off[30]) + 13 + at   # past the soft clip
        q_max = 43
        if what == "quality":
            b.seq[j], b.qual[j] = 15, q_max
            check(s, q_max)
            b.seq[j] = 4
        elif what == "reference":
            p = int(b.pos[30]) + 20 + at
            b.seqs[0] = b.seqs[0][:p] + b"R" + b.seqs[0][p + 1:]
            b.c_seqs[0] = b.seqs[0]
        else:
            b.seq[j] = what
        b.x1[30] = 1
        args = B.api.make_error_count_args(s, quality_max=q_max)
        with pytest.raises(B.BsqError):
            O.error_count(args)
        with pytest.raises(B.BsqError):
            B.api.error_count(s, quality_max=q_max)
