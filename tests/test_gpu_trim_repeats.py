"""Sequence and alignment trims where the repeat runs leave the words they are looked up in: sequences around
the 1,024-position blocks and 64-position words, periodic ones (units of 1 to 18 and 19) whose runs cross
them and pass 255 positions, and alignments whose edge repeats end at, before and behind 32 bases, with
clips and N bases; against a plain scan."""
import numpy as np
import pytest

import breseq_amd as B
from aln_builder import Built, BuiltSample

pytestmark = pytest.mark.gpu


def extent(s, p, n):
    """Longest perfect tandem repeat of a unit of 1..18 at p, at least 1 (calculate_trims.cpp:44-56)."""
    best = 1
    for u in range(1, 19):
        num = 1
        while p + u * num + u <= n and s[p:p + u] == s[p + u * num:p + u * num + u]:
            num += 1
        if num > 1:
            best = max(best, num * u)
    return best


def trims(s):
    n = len(s)
    left, right = np.zeros(n, np.int64), np.zeros(n, np.int64)
    for p in range(n):
        m = min(extent(s, p, n), 255)
        x = np.arange(p, min(n, p + m))
        right[x] = np.maximum(right[x], x - p + 1)
        left[x] = np.maximum(left[x], m - (x - p))
    return left, right


def text(kind, n, seed=0):
    rng = np.random.default_rng(seed + n)
    s = "".join(rng.choice(list("ACGT"), n))
    if kind == "random":
        return s
    if kind == "low":   # two letters: many short repeats
        return "".join(rng.choice(list("AC"), n))
    unit = s[:kind]
    p = (unit * (n // kind + 1))[:n]
    return s[:n // 5] + p[n // 5:n - n // 7] + s[n - n // 7:]


@pytest.mark.parametrize("kind", ["random", "low", 1, 2, 7, 18, 19])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 300, 1023, 1024, 1025, 2200])
def test_sequence_trims(kind, n):
    print("[gpu] trims of", kind, n, flush=True)
    s = text(kind, n)
    left, right = trims(s)
    got = B.calculate_trims(s)
    assert np.array_equal(np.asarray(got[0]), left) and np.array_equal(np.asarray(got[1]), right)


@pytest.mark.parametrize("m", [1, 18, 31, 32, 33, 37, 64, 90])
def test_alignment_trims(m):
    print("[gpu] alignment trims, spans of", m, flush=True)
    rng = np.random.default_rng(m)
    ref = text("random", 600, 5)
    left, right = trims(ref)
    reads, want = [], []
    for i in range(160):
        pos = int(rng.integers(0, 600 - m))
        kind = i % 6
        s = ref[pos:pos + m]
        if kind == 1:
            s = (s[:int(rng.integers(1, 20))] * 90)[:m]                      # periodic throughout
        elif kind == 2:
            u = s[:int(rng.integers(1, 5))]
            s = (u * int(rng.integers(2, 9)) + s)[:m]                        # a repeat at the start
        elif kind == 3:
            u = s[:int(rng.integers(1, 12))]
            s = (s + u * int(rng.integers(2, 9)))[-m:]                       # at the end
        elif kind == 4:
            s = "".join(c if rng.random() < 0.9 else "N" for c in s)
        a, b = (int(rng.integers(0, 5)), int(rng.integers(0, 5))) if i % 2 else (0, 0)
        cigar = ("%dS" % a if a else "") + "%dM" % m + ("%dS" % b if b else "")
        reads.append(dict(pos=pos, cigar=cigar, seq="A" * a + s + "C" * b, flag=16 if rng.random() < 0.5 else 0))
        # a repeat read backwards matches where the reversed sequence does
        want.append((max(left[pos], extent(s, 0, m)) + a, max(right[pos + m - 1], extent(s[::-1], 0, m)) + b))
    order = sorted(range(len(reads)), key=lambda k: reads[k]["pos"])
    sess = B.Session().load(BuiltSample(Built([("t0", ref)], [reads[k] for k in order])))
    try:
        xl, xr = sess.alignment_trims()
    finally:
        sess.close()
    assert [(int(l), int(r)) for l, r in zip(xl, xr)] == [tuple(int(v) for v in want[k]) for k in order]
