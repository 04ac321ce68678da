"""Scans by minimizer bins (the default for k = 20..31) against the radix path
on the same reads: labels, plan, per-scan counts, at the sizes where the bins
can go wrong -- every k they take, reads at and just past k, 'N's at record
ends, runs past a bin, one k-mer alone (the first-run quirk), many dead reads
and a few live ones, letters the bins leave to the radix path -- and batches."""
import numpy as np
import pytest

import metapart_amd as mp

FIELDS = ("tuples", "bad_labels", "zeroed_runs", "evaluated_runs", "quirk_segments")


def _fastq(seqs):
    return np.frombuffer("".join("@r%d\n%s\n+\n%s\n" % (i, s, "I" * len(s)) for i, s in enumerate(seqs)).encode(),
                         dtype=np.uint8).copy()


def _run(buf, C, K, S, T, **kw):
    with mp.Context(k=K, **kw) as ctx:
        ctx.load(buf, mp.index_buffer(buf, C))
        r = mp.partition(ctx, S=S, T=T, want_parent=True, build_output=False)
        return r, [[s[f] for f in FIELDS] for s in r.scans], [s["ms_sort_gen"] == 0 for s in r.scans]  # a radix scan times its generating pass


def _same(buf, C, K, S, T, bins=True):
    a, sa, pa = _run(buf, C, K, S, T)
    b, sb, pb = _run(buf, C, K, S, T, sort_digit_bits=7)  # a digit width asks for the radix sort
    assert not any(pb)
    if bins is not None:
        assert all(p == bins for p in pa), pa
    assert sa == sb
    assert np.array_equal(a.parent, b.parent)
    assert np.array_equal(a.W, b.W)
    return a


@pytest.mark.gpu
@pytest.mark.parametrize("K", list(range(20, 32)))
def test_every_k_equals_radix(K):
    print("gpu bins k", K, flush=True)
    buf = mp.synth(0, n_reads=6000, seed=300 + K, read_len_min=K - 3, read_len_max=K + 90, n_rate=0.004)
    _same(buf, 4, K, 1, 1 + K % 3)


@pytest.mark.gpu
def test_a_scan_by_bins_reports_no_radix_pass():
    print("gpu bins stats", flush=True)
    buf = mp.synth(0, n_reads=6000, seed=12, read_len=100)
    with mp.Context(k=31) as ctx:
        ctx.load(buf, mp.index_buffer(buf, 4))
        r = mp.partition(ctx, build_output=False)
        ctx.batch_load([buf, buf])
        _, st, _ = ctx.batch_partition()
    for s in (r.scans[0], st.as_dict()):
        for f in ("sort_passes", "ms_sort_pass_avg", "ms_sort_hist", "ms_sort_gen", "sort_local_moved", "ms_sort_count",
                  "sort_graph", "parts"):
            assert s[f] == 0, f
        assert s["ms_sort_local"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(2, 1), (3, 2), (1, 16)])
def test_scans_and_segments_equal_radix(S, T):
    print("gpu bins scans, segments", S, T, flush=True)
    _same(mp.synth(0, n_reads=20000, seed=77, read_len=120), 16, 27, S, T)


@pytest.mark.gpu
def test_many_scans_keep_to_the_bins_table():
    # 32 scans of 150 k shallow reads: a record holds a third of a window in the scan's range, and without those
    # that hold none every bin fits bin_runs
    print("gpu bins, 32 scans", flush=True)
    buf = mp.synth(0, n_reads=150000, seed=78, read_len=150, n_genomes=40, genome_len_min=500000, genome_len_max=1000000)
    a = _same(buf, 32, 31, 32, 1)
    assert [s["sort_long_groups"] for s in a.scans] == [0] * 32


@pytest.mark.gpu
@pytest.mark.parametrize("reads,S", [(60000, 2), (60000, 8), (200000, 16)])
def test_budgets_that_hold_the_radix_path_hold_the_bins(reads, S):
    # budgets from what the radix path held up to where bins fit too: a scan the bins cannot hold goes by radix
    # passes, and the pair step and the writer get their room, on a ctx's first run and on its second
    print("gpu bins budget", reads, S, flush=True)
    buf = mp.synth(0, n_reads=reads, read_len=150, seed=5, n_genomes=40, genome_len_min=50000, genome_len_max=300000)

    def run(budget, **kw):
        with mp.Context(k=31, hbm_budget=budget, **kw) as ctx:
            for _ in range(2):
                ctx.load(buf, mp.index_buffer(buf, 16))
                r = mp.partition(ctx, S=S, want_parent=True)
                assert not budget or ctx.device_bytes <= budget
            return r, ctx.device_bytes

    want, held = run(0, sort_digit_bits=7)
    for f in (1.0, 1.05, 1.1, 1.2, 1.3, 2.0):
        got, _ = run(int(held * f))
        assert np.array_equal(got.parent, want.parent) and np.array_equal(got.W, want.W) and got.out_bytes == want.out_bytes


@pytest.mark.gpu
@pytest.mark.parametrize("n,reads,L,K", [(3, 300, 100, 31), (8, 4000, 150, 31), (4, 60000, 45, 31), (1, 200000, 100, 21)])
def test_budgets_that_hold_a_radix_batch_hold_the_bins(n, reads, L, K):
    print("gpu bins batch budget", n, reads, L, K, flush=True)
    bufs = [mp.synth(0, n_reads=reads, read_len=L, seed=5 + i, n_genomes=10, genome_len_min=50000, genome_len_max=300000)
            for i in range(n)]

    def run(budget, **kw):
        with mp.Context(k=K, hbm_budget=budget, **kw) as ctx:
            for _ in range(2):
                ctx.batch_load(bufs)
                res, _, _ = ctx.batch_partition()
                nb = ctx.batch_write(None)
            return np.concatenate([ctx.batch_parent(i) for i in range(n)]), [list(map(int, r["W"])) for r in res], nb, \
                ctx.device_bytes

    want = run(0, sort_digit_bits=7)
    for f in (1.0, 1.05, 1.1, 1.3, 2.0):
        got = run(int(want[3] * f))
        assert np.array_equal(got[0], want[0]) and got[1:3] == want[1:3]


@pytest.mark.gpu
def test_records_at_read_and_step_ends():
    # reads of k - 1 .. k + 2 bases and of every length around a step's 960
    # positions, 'N' first, last, beside and between windows
    print("gpu bins record ends", flush=True)
    rng = np.random.default_rng(5)
    K = 31
    base = "".join("ACGT"[i] for i in rng.integers(0, 4, 4000))
    seqs = []
    for i in range(3000):
        L = [K - 1, K, K + 1, K + 2, 60, 64, 96, 240, 300, 20][i % 10]
        o = int(rng.integers(0, 4000 - 330))
        s = list(base[o:o + L])
        for p in {0: [], 1: [0], 2: [L - 1], 3: [L // 2], 4: [0, L - 1]}[i // 10 % 5]:
            s[p] = "N"
        if i % 7 == 0:
            s = [c.lower() if c != "N" else c for c in s]
        seqs.append("".join(s))
    _same(_fastq(seqs), 1, K, 1, 1)


@pytest.mark.gpu
def test_homopolymers_and_one_kmer():
    # one k-mer (the only run is the last, so the first-run quirk shows: the
    # radix path answers), the k-mer 0 alone beside others, and both ends
    print("gpu bins homopolymers", flush=True)
    a = _same(_fastq(["C" * 100] * 20), 1, 31, 1, 1, bins=False)
    assert a.scans[0]["quirk_segments"] == 1
    _same(_fastq(["A" * 90, "T" * 200] * 40 + ["ACGTTGCATCAGGATCAGCATTACGAGCATCGGACT"] * 4), 1, 25, 1, 1, bins=None)
    _same(_fastq(["AC" * 60, "CA" * 45, "AAC" * 40, "ACGT" * 30] * 200), 1, 31, 1, 1, bins=None)


@pytest.mark.gpu
def test_bins_past_the_table_and_a_few_live_reads():
    # a 500 bp genome at ~12000x (bins of far more windows and, by its errors,
    # k-mers than a table holds), then two reads of k + 1 bases that nothing filters
    print("gpu bins deep", flush=True)
    deep = mp.synth(0, n_reads=40000, n_genomes=1, genome_len_min=500, genome_len_max=500, read_len=150,
                    err_rate=0.01, seed=21)
    a = _same(deep, 4, 31, 1, 1)
    assert a.scans[0]["sort_long_groups"] > 0
    live = _fastq(["ACGGATTACCAGATTGCAGGCTTAACGGATCG", "TTGACCGATAGGACCAGTTTACCAGAGGATCC"])
    _same(np.concatenate([np.frombuffer(deep.tobytes(), dtype=np.uint8), live]), 1, 31, 1, 1, bins=None)


def _poly_g(n, err, seed):
    rng = np.random.default_rng(seed)
    seqs = []
    for _ in range(n):
        x = np.full(150, ord("G"), dtype=np.uint8)
        e = rng.random(150) < err
        x[e] = np.frombuffer(b"ACGT", dtype=np.uint8)[rng.integers(0, 4, int(e.sum()))]
        seqs.append(x.tobytes().decode())
    return _fastq(seqs)


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(1, 1), (2, 3)])
@pytest.mark.parametrize("deep", [False, True])
def test_piled_up_bins(deep, S, T):
    # a bin of many windows and few k-mers is visited a few times, not once per so many windows: 2 % poly-G reads
    # among others, and a 500 bp genome at 12000x, take less than a quarter of the radix path's time
    print("gpu bins piled up", deep, S, T, flush=True)
    if deep:
        buf = mp.synth(0, n_reads=40000, n_genomes=1, genome_len_min=500, genome_len_max=500, read_len=150,
                       err_rate=0.01, seed=22)
    else:
        buf = np.concatenate([np.frombuffer(mp.synth(0, n_reads=60000, read_len=150, seed=8).tobytes(), dtype=np.uint8),
                              _poly_g(1200, 0.003, 8)])
    a = _same(buf, 6, 31, S, T)
    b, _, _ = _run(buf, 6, 31, S, T, sort_digit_bits=7)
    assert all(s["sort_long_groups"] > 0 for s in a.scans)
    ms = [sum(s[f] for s in r.scans for f in ("ms_enumerate", "ms_sort", "ms_filter")) for r in (a, b)]
    assert ms[0] < ms[1] / 4, ms


def _amplicons(n, seed):
    """n reads that hold the 13-mer of the lowest minimizer hash between random bases: one bin of 19 n windows, as many k-mers"""
    mer = "".join("ACGT"[(0x2545F49 >> (24 - 2 * i)) & 3] for i in range(13))
    bases = np.frombuffer(b"ACGT", dtype=np.uint8)[np.random.default_rng(seed).integers(0, 4, (n, 137))]
    return _fastq([r[:60].tobytes().decode() + mer + r[60:].tobytes().decode() for r in bases])


@pytest.mark.gpu
def test_a_pile_of_distinct_kmers_goes_to_the_radix_path():
    print("gpu bins pile of distinct k-mers", flush=True)
    _same(_amplicons(14000, 3), 2, 31, 1, 1, bins=False)


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(1, 2), (2, 1), (2, 3)])
def test_scans_given_up_after_marks(S, T):
    # the same pile beside 200 k reads of several copies: three visits of it fit what the large bins may take, its
    # parts do not, so the scan is given up after reads were marked, and a later scan puts their flags back
    print("gpu bins given up", S, T, flush=True)
    buf = mp.synth(0, n_reads=200000, read_len=150, seed=31, n_genomes=20, genome_len_min=100000, genome_len_max=200000)
    both = np.concatenate([np.frombuffer(buf.tobytes(), dtype=np.uint8), _amplicons(12000, 4)])
    a = _same(both, 6, 31, S, T, bins=False)
    assert all(s["bad_labels"] > 0 for s in a.scans)


@pytest.mark.gpu
def test_other_letters_take_the_radix_path():
    print("gpu bins letters", flush=True)
    buf = np.frombuffer(mp.synth(0, n_reads=2000, seed=9, read_len=100).tobytes(), dtype=np.uint8).copy()
    nl = np.flatnonzero(buf == 10)
    buf[nl[40] + 50] = ord("Y")  # bit 3 set: its neighbour class is not in the 2-bit code
    _same(buf, 2, 27, 1, 1, bins=False)
    seqs = ["ACGGATTACCAGATTGCAGGCTTAACGGATCGAC"] * 10
    seqs[3] = ""
    _same(_fastq(seqs), 1, 27, 1, 1, bins=False)


@pytest.mark.gpu
def test_dump_after_bins_equals_radix():
    print("gpu bins dump", flush=True)
    buf = mp.synth(0, n_reads=5000, seed=4, read_len=90, n_rate=0.002)
    got = []
    for kw in ({}, {"sort_digit_bits": 7}):
        with mp.Context(k=25, **kw) as ctx:
            ctx.load(buf, mp.index_buffer(buf, 4))
            hist, _, _, _ = ctx.count()
            scan, thread = mp.plan_ranges(hist, 2, 2)
            out = []
            for s in range(2):
                ctx.scan(s, int(scan[s]), int(scan[s + 1]), thread[2 * s:2 * s + 3])
                out.append(ctx.dump_tuples())
            W, _ = ctx.finish()
            got.append((out, W, ctx.parent(), ctx.dump_tuples()))
    for x, y in zip(got[0][0] + [got[0][3]], got[1][0] + [got[1][3]]):
        assert np.array_equal(x, y)
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])


@pytest.mark.gpu
@pytest.mark.parametrize("reads,S,f", [(200000, 1, 1.05), (300000, 2, 1.05), (400000, 4, 1.1)])
def test_dump_in_the_radix_paths_budget(reads, S, f):
    # more windows than a scan holds the radix path's buffers for: a dump at the end sorts then, in a budget that the
    # radix path's dump goes through in, and leaves labels and files as they are
    print("gpu bins dump budget", reads, S, flush=True)
    buf = mp.synth(0, n_reads=reads, read_len=150, seed=5, n_genomes=40, genome_len_min=50000, genome_len_max=300000)

    def run(budget, **kw):
        with mp.Context(k=31, hbm_budget=budget, **kw) as ctx:
            ctx.load(buf, mp.index_buffer(buf, 16))
            r = mp.partition(ctx, S=S, want_parent=True)
            assert all(s["parts"] == 0 for s in r.scans)
            d = ctx.dump_tuples()
            assert np.array_equal(ctx.parent(), r.parent)
            assert ctx.write_partitions(None, 1, r.W, None) == r.out_bytes
            return r, d, ctx.device_bytes

    want, dump, held = run(0, sort_digit_bits=7)
    got, d, dev = run(int(held * f))
    assert dev <= held * f
    assert np.array_equal(d, dump) and np.array_equal(got.parent, want.parent) and got.out_bytes == want.out_bytes


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 70, 256])
def test_batch_equals_radix(n):
    print("gpu bins batch", n, flush=True)
    rng = np.random.default_rng(n)
    bufs = [mp.synth(0, n_reads=2 * int(rng.integers(1, 400)), seed=500 + i % 50, read_len=int(rng.integers(40, 150)))
            for i in range(n)]
    got = []
    for kw in ({}, {"sort_digit_bits": 7}):
        with mp.Context(k=31, **kw) as ctx:
            ctx.batch_load(bufs)
            res, st, _ = ctx.batch_partition()
            got.append(([[r[f] for f in ("reads", "tuples", "components", "largest")] + list(map(int, r["W"])) for r in res],
                        [getattr(st, f) for f in FIELDS], np.concatenate([ctx.batch_parent(i) for i in range(n)])))
    assert got[0][0] == got[1][0] and got[0][1] == got[1][1]
    assert np.array_equal(got[0][2], got[1][2])


@pytest.fixture(scope="module")
def big():
    """8.3 M reads of 150 bases, more than 1.2e9 bases, from 60 genomes at some 7x, their record starts known"""
    buf = mp.synth(0, n_reads=8300000, read_len=150, seed=41, n_genomes=60, genome_len_min=2000000, genome_len_max=4000000)
    yield buf
    buf.free()


def _front(buf, reads):
    """whole records from the front: `reads` of them, to an even number"""
    step = buf.nbytes // 8300000 + 2  # the longest record, or more
    v = buf.view()[:reads * step]
    return v[:int(np.flatnonzero(v == 10)[4 * reads - 1]) + 1]


@pytest.mark.gpu
@pytest.mark.parametrize("K", list(range(25, 32)))
def test_wide_minimizers_equal_radix(K, big):
    # more than 200 M bases: 15-base minimizers, whole scans and scans of part of the buckets
    print("gpu bins wide minimizers", K, flush=True)
    buf = _front(big, 1400000)
    for S, T in ((1, 1 + K % 4), (2 + K % 2, 1)):
        a = _same(buf, 12, K, S, T)
        assert sum(s["tuples"] for s in a.scans) == 1400000 * (151 - K)


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(1, 1), (2, 2)])
def test_large_inputs_equal_radix(S, T, big):
    # 13 cell bits, tiles of so many steps that records move in the larger batches
    print("gpu bins large", S, T, flush=True)
    a = _same(big.view(), 16, 31, S, T)
    assert sum(s["tuples"] for s in a.scans) == 8300000 * 120


@pytest.mark.gpu
def test_large_batch_equals_radix(big):
    print("gpu bins large batch", flush=True)
    v = big.view()
    cut = [0] + [len(_front(big, n)) for n in (2, 700000, 5000000)] + [big.nbytes]
    bufs = [v[a:b] for a, b in zip(cut, cut[1:])]
    got = []
    for kw in ({}, {"sort_digit_bits": 7}):
        with mp.Context(k=31, **kw) as ctx:
            ctx.batch_load(bufs)
            res, st, _ = ctx.batch_partition()
            assert (st.ms_sort_gen == 0) == (not kw)
            got.append(([[r[f] for f in ("reads", "tuples", "components", "largest")] + list(map(int, r["W"])) for r in res],
                        [getattr(st, f) for f in FIELDS], [ctx.batch_parent(i) for i in range(len(bufs))]))
    assert got[0][:2] == got[1][:2]
    assert all(np.array_equal(a, b) for a, b in zip(got[0][2], got[1][2]))
