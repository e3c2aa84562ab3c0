"""The work that users of the pileup-scoring engine have it do, as measurable cases.

Six kinds of call, all through breseq_amd's public entry points:

  pipeline       Session.pipeline on a sample that is resident on the GPU: error_count, the
                 coverage-distribution fit, identify_mutations (breseq's stages 07-08)
  serve          Session.load of an in-memory sample into a kept session, then the pipeline: what a
                 server does for each request
  preprocess     error_count of the preprocess stage (coverage and read starts, no error table)
  cov_table      BAM2COV coverage table of one region
  seq_trims      calculate_trims of one reference sequence
  aln_trims      XL / XR of every alignment of a resident sample

Samples come from the package's own seeded generator.  Sizes are those of the benchmark workloads
(breseq_amd.workloads), of the batched mix (breseq_amd.batch.mixed_jobs: lengths from 50 kb up,
coverage 20-300x, reads of 36, 100 and 150 bases) and of the tests (2x300 bp pairs, columns thousands
of reads deep).
"""
import math

import numpy as np

import breseq_amd as B
from breseq_amd import api, workloads

DP_SETS = [workloads.DP_SET]
QUALITY_MAX = 42   # the generated qualities end at 41; breseq passes max_qual + 1 of its summary


def _sample_case(name, kind, ref_length, read_length, coverage, paired, mode="consensus", **more):
    c = dict(name=name, kind=kind, ref_length=ref_length, read_length=read_length, coverage=coverage, paired=paired,
             mode=mode, gc=0.508, qual_mean=34, qual_sd=5, n_snps=max(2, ref_length // 9200),
             n_indels=max(1, ref_length // 92000), freq_min=1.0, freq_max=1.0, missing_edge_reads=6,
             n_missing=3 if ref_length >= 400000 and kind != "aln_trims" else 0)
    c.update(more)
    return c


def listed():
    poly = dict(mode="polymorphism", qual_mean=33, qual_sd=6, freq_min=0.01, freq_max=0.5)
    return [
        # the smallest sample: a phage-sized genome at low coverage, short single-end reads; launches,
        # copies and the host's own work are all of its time
        _sample_case("pipeline_48k_36bp_20x", "pipeline", 48502, 36, 20.0, False, gc=0.5, qual_mean=32, qual_sd=6),
        # 100,000 single-end reads of 100 bases on the same genome (the first benchmark workload)
        _sample_case("pipeline_48k_100bp_206x", "pipeline", 48502, 100, 100000 * 100 / 48502, False, gc=0.5, qual_mean=32,
                     qual_sd=6, n_snps=20, n_indels=2),
        # a bacterial clone: 4.6 Mb at 100x of 2x150 pairs with discordant pairs (the headline workload)
        _sample_case("pipeline_4600k_150bp_100x", "pipeline", 4600000, 150, 100.0, True, n_snps=500, n_indels=50),
        # a mixed population: 1 Mb at 300x in polymorphism mode, variants at 1-50%
        _sample_case("pipeline_poly_1000k_150bp_300x", "pipeline", 1000000, 150, 300.0, True, n_snps=390, n_indels=43,
                     missing_edge_reads=12, **poly),
        # old short-read data: 36-base reads, an odd genome length
        _sample_case("pipeline_2047k_36bp_83x", "pipeline", 2047303, 36, 83.0, False),
        # long paired reads, at an odd length
        _sample_case("pipeline_701k_300bp_57x", "pipeline", 701401, 300, 57.0, True),
        # a plasmid or amplicon sequenced very deeply, columns of some 3,000 reads
        _sample_case("pipeline_poly_20k_150bp_3001x", "pipeline", 20011, 150, 3001.0, True, n_snps=20, n_indels=4, **poly),
        # one served request: the load of a new sample into a kept session, then the pipeline
        _sample_case("serve_1300k_150bp_90x", "serve", 1300031, 150, 90.0, True),
        # the preprocess stage's error_count of a medium sample
        _sample_case("preprocess_2300k_100bp_40x", "preprocess", 2300011, 100, 40.0, False),
        # BAM2COV of a whole genome at the default resolution
        _sample_case("cov_table_1000k_150bp_100x", "cov_table", 1000000, 150, 100.0, True, start=0, end=0, resolution=600,
                     total_only=False, per_read_group=False),
        # the trims of a bacterial reference
        dict(name="seq_trims_4600k", kind="seq_trims", ref_length=4600000, gc=0.508),
        # the trim tags of every alignment of a sample
        _sample_case("aln_trims_1000k_150bp_60x", "aln_trims", 1000003, 150, 60.0, True),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pipeline"] * 6 + ["serve", "preprocess", "cov_table", "seq_trims", "aln_trims"])
    gc = round(rng.uniform(0.35, 0.65), 3)
    if kind == "seq_trims":
        return dict(kind=kind, ref_length=int(_log_uniform(rng, 5000, 4600000)) | 1, gc=gc)
    poly = kind in ("pipeline", "serve") and rng.random() < 0.4
    ref_length = int(_log_uniform(rng, 20000, 1000000 if poly or kind in ("serve", "cov_table", "aln_trims") else 4600000))
    # aligned bases: no drawn case costs more than the listed ones of its kind
    most = dict(pipeline=4.0e8, serve=1.0e8, preprocess=9.0e7, cov_table=1.0e8, aln_trims=6.0e7)[kind]
    if poly:
        most = 6.0e7 if ref_length < 60000 else 1.0e8
    read_length = rng.choice([36, 100, 150, rng.randrange(36, 301)])
    deepest = min(3000.0 if ref_length < 60000 else 300.0, most / ref_length)
    coverage = round(_log_uniform(rng, min(15.0, deepest), deepest), 1)
    paired = read_length >= 100 and rng.random() < 0.6
    more = dict(gc=gc, qual_mean=rng.randrange(28, 37), qual_sd=rng.randrange(3, 8))
    if poly:
        more.update(freq_min=0.01, freq_max=0.5)
    if kind == "cov_table":
        span = int(_log_uniform(rng, 1000, ref_length))
        start = 1 + rng.randrange(0, ref_length - span + 1)
        more.update(start=start, end=start + span - 1, resolution=rng.choice([600, 600, 100, 0]),
                    total_only=rng.random() < 0.3, per_read_group=rng.random() < 0.3)
        if more["resolution"] == 0 and span > 20000:
            more["resolution"] = 600
    c = _sample_case("", kind, ref_length, read_length, coverage, paired, "polymorphism" if poly else "consensus", **more)
    del c["name"]
    return c


def _simulate(c, seed):
    s = B.Sample.simulate(seed=1 + seed % (1 << 31), ref_length=c["ref_length"], gc=c["gc"], read_length=c["read_length"],
                          coverage=c["coverage"], paired=c["paired"], insert_mean=max(350, 2 * c["read_length"] + 50),
                          insert_sd=50, qual_mean=c["qual_mean"], qual_sd=c["qual_sd"], qual_min=2, qual_max=41,
                          n_snps=c["n_snps"], n_indels=c["n_indels"], indel_max=5, variant_freq_min=c["freq_min"],
                          variant_freq_max=c["freq_max"], redundant_fraction=0.01, mapq=42,
                          discordant_fraction=0.002 if c["paired"] else 0.0, n_junctions=40 if c["paired"] else 0,
                          n_missing=c["n_missing"], missing_length=400 if c["n_missing"] else 0,
                          missing_edge_reads=c["missing_edge_reads"] if c["n_missing"] else 0)
    return s


def _random_reference(c, seed):
    """A random sequence of the given GC with homopolymers and tandem repeats every few hundred bases,
    a few of them longer than the 255-base cap of a trim."""
    rng = np.random.default_rng(seed)
    n, gc = c["ref_length"], c["gc"]
    s = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), n, p=[(1 - gc) / 2, gc / 2, gc / 2, (1 - gc) / 2])
    k = max(1, n // 400)
    at = rng.integers(0, n, k)
    unit = rng.integers(1, 19, k)
    copies = rng.integers(2, 9, k)
    copies[rng.random(k) < 0.002] = 320
    for p, u, m in zip(at.tolist(), unit.tolist(), copies.tolist()):
        run = np.tile(s[p:p + u], m)[: n - p]
        s[p:p + run.size] = run
    return s.tobytes().decode()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "seq_trims":
        return dict(kind=kind, seq=_random_reference(case, seed))
    sample = _simulate(case, seed)
    session = B.Session().load(sample)
    mode = B.POLYMORPHISM if case["mode"] == "polymorphism" else B.CONSENSUS
    dp = api.dp_settings(DP_SETS, seed=workloads.DP_SEED) if case["paired"] else None
    st = dict(kind=kind, sample=sample, session=session, mode=mode, dp=dp)
    # outputs whose length depends on the data go into buffers of the state, zeros after their end
    n, depth = case["ref_length"], case["coverage"]
    entries = 200 + 40 * (case["n_snps"] + case["n_indels"]) + n * min(1.0, math.exp(-depth / 5.0))
    st["out"] = dict(histogram=_Padded(int(8 * depth) + 512, np.uint32), gd=_Padded(int(400 * entries) + 65536, np.uint8),
                     dp=_Padded(1 << 20, np.uint8), rates_text=_Padded(1 << 18, np.uint8))
    if kind == "cov_table":
        st["table"] = {k: case[k] for k in ("start", "end", "resolution", "total_only", "per_read_group")}
        span = case["end"] - case["start"] + 1 if case["end"] else n
        rows = span if case["resolution"] == 0 else min(span, 2 * case["resolution"] + 2 * int(case["read_length"]))
        st["out"] = dict(table=_Padded(200 * rows + 65536, np.uint8))
    return st


class _Padded:
    """A buffer of fixed length that outputs of varying length are copied to; the rest stays zero."""

    def __init__(self, size, dtype):
        self.a, self.used = np.zeros(size, dtype=dtype), 0

    def put(self, v):
        if isinstance(v, str):
            v = np.frombuffer(v.encode(), dtype=np.uint8)
        self.a[:v.size] = v
        self.a[v.size:self.used] = 0
        self.used = v.size
        return self.a


def run(state):
    kind = state["kind"]
    if kind == "seq_trims":
        left, right = B.api.calculate_trims(state["seq"])
        return dict(left=left, right=right)
    session, out = state["session"], state.get("out")
    if kind == "cov_table":
        return dict(table=out["table"].put(session.coverage_table(**state["table"])))
    if kind == "aln_trims":
        xl, xr = session.alignment_trims()
        return dict(xl=xl, xr=xr)
    if kind == "preprocess":
        ec = session.error_count(do_errors=False, preprocess_stage=True, quality_max=QUALITY_MAX)
        return dict(histogram=out["histogram"].put(ec.histograms[0]), no_pos_hash_pr=ec.no_pos_hash_pr)
    if kind == "serve":
        session.load(state["sample"])
    ec, summaries, gd, dp = session.pipeline(mode=state["mode"], dp=state["dp"], ec_kw=dict(quality_max=QUALITY_MAX))
    return dict(histogram=out["histogram"].put(ec.histograms[0]), counts=ec.counts, log10_prob=ec.log10_prob,
                rates_table=ec.rates_table, rates_text=out["rates_text"].put(ec.rates_text),
                summaries=[list(s.values()) for s in summaries], gd=out["gd"].put(gd), dp=out["dp"].put(dp))


def work(case):
    """Each base, quality and alignment record (24 bytes) read once, the reference read once, the
    outputs written once; the operations are the five likelihood sums and the two counts of a base."""
    kind, n = case["kind"], case["ref_length"]
    if kind == "seq_trims":
        return dict(bytes=3 * n, flops=18 * n)   # a comparison per position and repeat unit
    bases = n * case["coverage"]
    reads = bases / case["read_length"]
    if kind == "preprocess":
        return dict(bytes=24 * reads + n, flops=2 * reads)
    if kind == "cov_table":
        span = case["end"] - case["start"] + 1 if case["end"] else n
        rows = span if case["resolution"] == 0 else min(span, case["resolution"])
        deep = case["coverage"] * rows * (2 if case["per_read_group"] else 1)
        return dict(bytes=24 * min(reads, deep) + 40 * rows, flops=2 * deep)
    if kind == "aln_trims":
        return dict(bytes=32 * reads + 2 * 18 * reads + n, flops=36 * reads + 18 * n)
    # a served sample's arrays are read on the host and written to the device as well
    return dict(bytes=(2 * bases + 24 * reads + n) * (3 if kind == "serve" else 1), flops=7 * bases)


def tolerance(case):
    """Counts, trims and texts are whole numbers and bytes: the same.  The printed numbers and the
    64-bit tables come from exact counts and ordered 64-bit sums; a different libm or order of a
    short sum moves a table entry by a few units in the last place (measured against exact(): at
    most 2e-16, stated with room for the logarithms of another library)."""
    if case["kind"] in ("seq_trims", "aln_trims", "cov_table"):
        return "exact"
    return dict(rel=1e-14)


def _laplace(counts, S, Q):
    """log10((count + 1) / (sum over the observed classes + 5)) per read set, reference class and quality."""
    c = counts.reshape(Q, 5, 5, S).astype(np.float64)   # quality, observed, reference, read set
    return (np.log10(c + 1.0) - np.log10(c.sum(axis=1, keepdims=True) + 5.0)).reshape(-1)


def _six_digits(v):
    return np.array([float("%g" % x) for x in v])


_COMP = np.array([3, 2, 1, 0, 4])


def _count_table(sample, S, Q):
    """breseq's covariate counts of a generated sample: reads of A, C, G, T and N, references of A, C, G, T
    (count_alignment_position, error_count.cpp:854-986)."""
    a = sample.arrays()
    refs = [np.searchsorted(np.frombuffer(b"ACGT", dtype=np.uint8), np.frombuffer(s.encode(), dtype=np.uint8))
            for _, s in sample.reference_sequences()]
    ref = np.concatenate([np.append(r, 9) for r in refs])   # one column after each target
    offs = np.concatenate([[0], np.cumsum([r.size + 1 for r in refs])])
    code = np.full(16, 9)
    code[[1, 2, 4, 8]] = [0, 1, 2, 3]
    cig, coff, soff = a["cigar"], a["cigar_off"], a["seq_off"]
    op, ln = cig & 15, (cig >> 4).astype(np.int64)
    n = len(a["pos"])
    read_of = np.repeat(np.arange(n), np.diff(coff))
    in_ref, in_query = np.isin(op, [0, 2, 3, 7, 8]), np.isin(op, [0, 1, 4, 7, 8])

    def starts(take):   # start of each operation within its read
        c = np.concatenate([[0], np.cumsum(np.where(take, ln, 0))])
        return c[:-1] - c[coff[read_of]]

    rev = (a["flag"] & 16) != 0
    rset = np.where((a["flag"] & 128) != 0, 1, 0) if S > 1 else np.zeros(n, dtype=np.int64)
    rset = rset.astype(np.int64)
    x0 = offs[a["tid"][read_of]] + a["pos"][read_of] + starts(in_ref)
    y0 = starts(in_query)
    # last aligned query base: soft clips at the end excluded
    qlen = np.diff(soff)
    last_op = coff[1:] - 1
    qe0 = qlen - 1 - np.where(op[last_op] == 4, ln[last_op], 0)
    used = np.isin(op, [0, 7, 8]) & (a["x1"][read_of] <= 1) & ((a["flag"][read_of] & 4) == 0) & (ln > 0)
    runs = np.nonzero(used)[0]
    # the indel that follows a run
    nxt = np.minimum(runs + 1, len(op) - 1)
    has = runs + 1 < coff[read_of[runs] + 1]
    indel = np.where(has & (op[nxt] == 2), -ln[nxt], np.where(has & (op[nxt] == 1), ln[nxt], 0))
    out = np.zeros(25 * S * Q, dtype=np.int64)

    def add(rs, r, o, q):
        out[:] += np.bincount(rs + S * r + 5 * S * o + 25 * S * q, minlength=out.size)

    R, L = read_of[runs], ln[runs]
    k = np.repeat(np.arange(runs.size), L)
    d = np.arange(k.size) - np.repeat(np.cumsum(L) - L, L)
    rd, y = R[k], y0[runs][k] + d
    x = x0[runs][k] + d
    seq, qual = a["seq"], a["qual"].astype(np.int64)
    at = soff[rd] + y
    flip = rev[rd]

    def fold(cls, flags):
        return np.where(flags, _COMP[np.minimum(cls, 4)], cls)

    acgt = code[seq[at]] < 4
    add(rset[rd][acgt], fold(ref[x], flip)[acgt], fold(code[seq[at]], flip)[acgt], qual[at][acgt])
    # '..' pairs: the next base in read direction, unless an indel follows or the aligned part ends
    lastq = y0[runs] + L - 1
    end = np.where(indel != 0, np.minimum(qe0[R], lastq), qe0[R])
    at2 = np.minimum(at + np.where(flip, 0, 1), qual.size - 1)
    pair = (y < end[k]) & (code[seq[at2]] < 4)
    q2 = qual[at2]
    four = np.full(int(pair.sum()), 4)
    add(rset[rd][pair], four, four, q2[pair])
    # one-base deletions and insertions after the run's last base
    for want in (-1, 1):
        e = np.nonzero(indel == want)[0]
        if not e.size:
            continue
        re, fl = R[e], rev[R[e]]
        p, qp = x0[runs][e] + L[e] - 1, lastq[e]
        if want == -1:
            at1 = soff[re] + qp + np.where(fl, 0, 1)
            ok = code[seq[at1]] < 4
            add(rset[re][ok], fold(ref[p + 1], fl)[ok], np.full(int(ok.sum()), 4), qual[at1][ok])
        else:
            at1 = soff[re] + qp + 1
            ok = (qp + 1 <= qe0[re]) & (code[seq[at1]] < 4)
            add(rset[re][ok], np.full(int(ok.sum()), 4), fold(code[seq[at1]], fl)[ok], qual[at1][ok])
    return out


def exact(case, seed):
    """The error table in 64 bits from counts made with numpy; None where the sample is too large for
    that.  The other outputs are whole numbers, texts, or the fit of the coverage distribution."""
    if case["kind"] not in ("pipeline", "serve") or case["ref_length"] * case["coverage"] > 2.5e7:
        return None
    sample = _simulate(case, seed)
    S, Q = (2 if case["paired"] else 1), QUALITY_MAX
    counts = _count_table(sample, S, Q)
    table = _laplace(counts, S, Q)
    return dict(histogram=None, counts=counts, log10_prob=table, rates_table=_six_digits(table), rates_text=None,
                summaries=None, gd=None, dp=None)
