"""Timed cases of the partitioning path, through the package's public calls.

Every case is one program a user of this package writes: FASTQ bytes in hand
(in host memory, as a file read gives them, or already in HBM, as a pipeline
on the device leaves them), a context or a server that the program keeps, and
one pass from the bytes to the labels, the plan and the partitioned streams.

Reads come from random genomes as the package's own generator makes them
(per-genome GC fraction in U(0.3, 0.7), log-normal abundances, both strands,
substitutions, some 'N's), drawn on the GPU so that inputs are made quickly.

Every output is a whole number (labels, plan, counts): there is nothing that
64-bit arithmetic would say better, so exact() has no values to give.
"""
import ctypes
import math

import numpy as np
import torch

import metapart_amd as mp

# what a case says beside its name:
#   kind       partition | count | noalloc | batch | serve
#   reads      records of the input; reads_min, reads_max: of a batch's samples or of the jobs
#   len_min, len_max   read lengths; k, chunks, S (scans), T (segments)
#   genomes, genome_len   genomes and their mean length; sigma: spread of their abundances
#   err, n_rate   substitutions and 'N's per base
#   host       the FASTQ bytes lie in host memory, and the pass uploads them


def listed():
    return [
        # A first try of the tools on a handful of reads (the size of the sample file that ships with the
        # tests): every launch and every wait counts.
        dict(name="try_2k", kind="partition", reads=2500, len_min=100, len_max=100, k=27, chunks=4, S=1, T=1,
             min3=False, paired=False, genomes=4, genome_len=20000, sigma=0.5, err=0.01, n_rate=0.0, host=True,
             write=True),
        # One amplicon-sized sample with trimmed reads and 'N's, in two scans of three segments.
        dict(name="trimmed_30k_S2T3", kind="partition", reads=30002, len_min=50, len_max=160, k=25, chunks=6, S=2,
             T=3, min3=False, paired=False, genomes=10, genome_len=60000, sigma=1.0, err=0.01, n_rate=0.002,
             host=True, write=True),
        # The mean job of a request loop, uploaded and partitioned on its own; labels only.
        dict(name="job_529k", kind="partition", reads=529000, len_min=150, len_max=150, k=31, chunks=1, S=1, T=1,
             min3=False, paired=False, genomes=60, genome_len=1750000, sigma=1.0, err=0.01, n_rate=0.0, host=True,
             write=False),
        # Interleaved read pairs with a short k, two segments.
        dict(name="pairs_1m_k27", kind="partition", reads=1000000, len_min=125, len_max=125, k=27, chunks=16, S=1,
             T=2, min3=False, paired=True, genomes=40, genome_len=1000000, sigma=1.0, err=0.01, n_rate=0.0005,
             host=False, write=True),
        # The first reads of a large share in four bucket scans, as a small memory budget asks for.
        dict(name="share_2m_S4", kind="partition", reads=2000000, len_min=150, len_max=150, k=31, chunks=64, S=4,
             T=1, min3=False, paired=False, genomes=100, genome_len=2000000, sigma=1.5, err=0.01, n_rate=0.0,
             host=False, write=True),
        # A deep sample of quality-trimmed reads at k = 21 in four segments: k-mers of many copies.
        dict(name="deep_2m_k21_T4", kind="partition", reads=2222222, len_min=60, len_max=125, k=21, chunks=16, S=1,
             T=4, min3=False, paired=False, genomes=30, genome_len=150000, sigma=1.0, err=0.005, n_rate=0.001,
             host=False, write=True),
        # The 3-minimizer variant.
        dict(name="min3_4m", kind="partition", reads=4000000, len_min=150, len_max=150, k=31, chunks=16, S=1, T=1,
             min3=True, paired=False, genomes=60, genome_len=3000000, sigma=0.0, err=0.01, n_rate=0.0, host=False,
             write=True),
        # The headline path: a metagenome of a hundred genomes, resident in HBM, one scan, one segment.
        dict(name="plain_12m", kind="partition", reads=12000000, len_min=150, len_max=150, k=31, chunks=16, S=1, T=1,
             min3=False, paired=False, genomes=120, genome_len=3000000, sigma=0.0, err=0.01, n_rate=0.0, host=False,
             write=True),
        # The histogram tool: bucket counts per chunk of a file's bytes.
        dict(name="count_1m", kind="count", reads=1000000, len_min=150, len_max=150, k=31, chunks=16, min3=False,
             genomes=50, genome_len=1000000, sigma=0.5, err=0.01, n_rate=0.0005),
        # The same counts inside a request loop that may not allocate.
        dict(name="noalloc_60k", kind="noalloc", reads=60000, len_min=100, len_max=150, k=31, chunks=4, min3=False,
             genomes=20, genome_len=200000, sigma=0.5, err=0.01, n_rate=0.0005),
        # Many samples of one study in one launch sequence.
        dict(name="batch_24", kind="batch", samples=24, reads_min=10000, reads_max=400000, len_min=100, len_max=150,
             k=31, min3=False, genomes=40, genome_len=150000, sigma=1.0, err=0.01, n_rate=0.0),
        # A queue of jobs of several sizes for the request loop.
        dict(name="serve_12", kind="serve", jobs=12, engines=3, reads_min=50000, reads_max=500000, len_min=150,
             len_max=150, k=31, min3=False, genomes=30, genome_len=500000, sigma=1.0, err=0.01, n_rate=0.0),
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _even(x):
    return max(2, int(x) // 2 * 2)


def draw(rng):
    kind = rng.choice(["partition"] * 7 + ["count", "noalloc", "batch", "serve"])
    k = rng.choice([21, 23, 25, 27, 29, 31, 31, 31, rng.randint(13, 32)])
    lmax = rng.randint(max(60, k + 10), 200)
    lmin = rng.choice([lmax, lmax, rng.randint(max(20, lmax // 3), lmax)])
    base = dict(kind=kind, k=k, len_min=lmin, len_max=lmax, min3=False, sigma=rng.choice([0.0, 0.5, 1.0, 1.5]),
                err=round(rng.uniform(0.002, 0.02), 4), n_rate=rng.choice([0.0, 0.0, 0.0005, 0.002]))

    def pool(reads):  # genomes for a mean depth between 2 and 60
        bases = reads * (lmin + lmax) / 2
        total = max(20000.0, bases / _log(rng, 2, 60))
        g = max(1, min(200, int(total / _log(rng, 20000, 3000000))))
        return dict(genomes=g, genome_len=int(total / g) + 1000)

    if kind == "partition":
        reads = _even(_log(rng, 2000, 5000000))
        min3 = rng.random() < 0.15
        S = 1 if min3 or reads < 50000 else rng.choice([1, 1, 1, 2, 3])
        T = 1 if reads < 20000 else rng.choice([1, 1, 2, 4])
        base.update(reads=reads, S=S, T=T, chunks=T * rng.choice([1, 3, 4, 8]), min3=min3,
                    paired=rng.random() < 0.2, host=rng.random() < 0.4, write=rng.random() < 0.8, **pool(reads))
    elif kind == "count":
        reads = _even(_log(rng, 5000, 2000000))
        base.update(reads=reads, chunks=rng.choice([1, 4, 7, 16, 32]), min3=rng.random() < 0.25, **pool(reads))
    elif kind == "noalloc":
        reads = _even(_log(rng, 2000, 50000))
        base.update(reads=reads, chunks=rng.randint(1, 8), min3=rng.random() < 0.25, **pool(reads))
    else:
        hi = _log(rng, 20000, 300000)
        base.update(reads_min=_even(hi / _log(rng, 2, 20)), reads_max=_even(hi), **pool(hi))
        if kind == "batch":
            base.update(samples=rng.randint(2, 40), min3=rng.random() < 0.15)
        else:
            base.update(jobs=rng.randint(2, 16), engines=rng.choice([1, 2, 3]))
    return base


# ---------------------------------------------------------------- inputs
_DEV = "cuda"


def _genomes(case, g):
    """(bases of all genomes in a row, first base and length of each, weights)"""
    n, mean = int(case["genomes"]), int(case["genome_len"])
    lens = (torch.rand(n, generator=g, device=_DEV, dtype=torch.float64) * mean + mean / 2).long() + 300
    first = torch.cumsum(lens, 0) - lens
    gc = torch.rand(n, generator=g, device=_DEV) * 0.4 + 0.3
    total = int(lens.sum())
    seq = torch.empty(total, dtype=torch.uint8, device=_DEV)
    of = torch.repeat_interleave(gc, lens)
    u = torch.rand(total, generator=g, device=_DEV)
    pick = torch.randint(0, 2, (total,), generator=g, device=_DEV, dtype=torch.uint8)
    seq = torch.where(u < of, torch.where(pick == 0, 67, 71), torch.where(pick == 0, 65, 84)).to(torch.uint8)
    w = torch.exp(torch.randn(n, generator=g, device=_DEV) * float(case["sigma"])) * lens
    return seq, first, lens, w


def _fastq(case, reads, seed):
    """(FASTQ bytes on the GPU, byte offset of every record and of the end)"""
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    seq, first, lens, w = _genomes(case, g)
    lmin, lmax, paired = int(case["len_min"]), int(case["len_max"]), bool(case.get("paired"))
    insert = max(lmax, 300) if paired else lmax
    acgt = torch.tensor([65, 67, 71, 84], dtype=torch.uint8, device=_DEV)
    comp = torch.arange(256, dtype=torch.uint8, device=_DEV)
    for a, b in ((65, 84), (67, 71), (71, 67), (84, 65)):
        comp[a] = b
    parts, sizes = [], []
    step = 1 << 19
    for a in range(0, reads, step):
        n = min(step, reads - a)
        frag = n // 2 if paired else n
        which = torch.multinomial(w.float(), frag, replacement=True, generator=g)
        room = torch.clamp(lens[which] - insert, min=1)
        at = first[which] + (torch.rand(frag, generator=g, device=_DEV, dtype=torch.float64) * room).long()
        back = torch.rand(frag, generator=g, device=_DEV) < 0.5
        if paired:  # mates from the two ends of a fragment, on opposite strands
            at = torch.stack([at, at + insert - lmax], 1).reshape(-1)
            back = torch.stack([back, ~back], 1).reshape(-1)
        col = torch.arange(lmax, device=_DEV)
        idx = at[:, None] + torch.where(back[:, None], lmax - 1 - col[None, :], col[None, :])
        s = seq[torch.clamp(idx, max=seq.numel() - 1)]
        del idx
        s = torch.where(back[:, None], comp[s.int()], s)
        u = torch.rand(s.shape, generator=g, device=_DEV)
        s = torch.where(u < float(case["err"]), acgt[torch.randint(0, 4, s.shape, generator=g, device=_DEV)], s)
        if float(case["n_rate"]) > 0:
            s = torch.where(u > 1.0 - float(case["n_rate"]), torch.full_like(s, 78), s)
        del u
        ids = torch.arange(a, a + n, device=_DEV)
        head = torch.empty((n, 12), dtype=torch.uint8, device=_DEV)
        head[:, 0], head[:, 1], head[:, 11] = 64, 114, 10
        for d in range(9):
            head[:, 10 - d] = (48 + ids // 10 ** d % 10).to(torch.uint8)
        plus = torch.tensor([10, 43, 10], dtype=torch.uint8, device=_DEV).expand(n, 3)
        end = torch.full((n, 1), 10, dtype=torch.uint8, device=_DEV)
        rows = torch.cat([head, s, plus, torch.full_like(s, 73), end], 1)
        if lmin < lmax:
            ln = torch.randint(lmin, lmax + 1, (n,), generator=g, device=_DEV)
            keep = col[None, :] < ln[:, None]
            one = torch.ones((n, 1), dtype=torch.bool, device=_DEV)
            rows = rows[torch.cat([one.expand(n, 12), keep, one.expand(n, 3), keep, one], 1)]
            sizes.append((16 + 2 * ln).cpu())
        else:
            rows = rows.reshape(-1)
            sizes.append(torch.full((n,), 16 + 2 * lmax))
        parts.append(rows)
    total = sum(p.numel() for p in parts)
    fq = torch.zeros(total + 64, dtype=torch.uint8, device=_DEV)
    o = 0
    for i, p in enumerate(parts):
        fq[o:o + p.numel()] = p
        o += p.numel()
        parts[i] = None
    start = np.concatenate([[0], np.cumsum(torch.cat(sizes).numpy())]).astype(np.uint64)
    del seq, rows, s
    torch.cuda.empty_cache()
    return fq, start


def _chunks(start, C):
    n = len(start) - 1
    return start[[n * c // C // 2 * 2 for c in range(C)] + [n]]


def _sizes(case, count):
    """Read counts of a batch's samples or of the jobs: log-uniform, the same for every seed of a case."""
    r = np.random.default_rng(count)
    x = np.exp(r.uniform(math.log(case["reads_min"]), math.log(case["reads_max"]), count))
    return [_even(v) for v in x]


def prepare(case, seed):
    c = dict(case)
    seed = int(seed) * 1000003 % (1 << 40)
    st = {"case": c}
    kind = c["kind"]
    if kind in ("partition", "count", "noalloc"):
        fq, start = _fastq(c, int(c["reads"]), seed)
        st["nbytes"] = int(start[-1])
        st["cofs"] = _chunks(start, int(c["chunks"]))
        if kind == "count" or c.get("host"):
            st["fq"] = fq[: st["nbytes"]].cpu().numpy()
        else:
            st["fq"] = fq
        if kind == "noalloc":
            C = int(c["chunks"])
            st["counts"] = np.zeros((C, mp.NBUCKETS + 2), dtype=np.uint32)
            st["reads"] = np.zeros(C, dtype=np.uint64)
        else:
            st["ctx"] = mp.Context(k=int(c["k"]), min3=bool(c["min3"]))
    elif kind == "batch":
        parts, ofs = [], [0]
        for i, n in enumerate(_sizes(c, int(c["samples"]))):
            fq, start = _fastq(c, n, seed + 1 + i)
            parts.append(fq[: int(start[-1])])
            ofs.append(ofs[-1] + int(start[-1]))
        st["fq"] = torch.cat(parts + [torch.zeros(64, dtype=torch.uint8, device=_DEV)])
        st["ofs"] = np.array(ofs, dtype=np.uint64)
        st["ctx"] = mp.Context(k=int(c["k"]), min3=bool(c["min3"]))
    else:
        st["jobs"] = []
        for i, n in enumerate(_sizes(c, int(c["jobs"]))):
            fq, start = _fastq(c, n, seed + 1 + i)
            st["jobs"].append(fq[: int(start[-1])].cpu().numpy())
        st["srv"] = mp.Server(k=int(c["k"]), engines=int(c["engines"]), hbm_budget=24 << 30)
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------- passes
def _whole(a):
    return np.asarray(a).view(np.int64)


def _load(st):
    if isinstance(st["fq"], np.ndarray):
        st["ctx"].load(st["fq"], st["cofs"])
    else:
        st["ctx"].load_device(st["fq"].data_ptr(), st["nbytes"], st["cofs"])


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "partition":
        _load(st)
        il = [0] * int(c["chunks"]) if c["paired"] else None
        r = mp.partition(st["ctx"], S=int(c["S"]), T=int(c["T"]), want_parent=True, il_start=il,
                         build_output=bool(c["write"]))
        whole = ("tuples", "bad_labels", "zeroed_runs", "evaluated_runs", "quirk_segments")
        return {"parent": _whole(r.parent), "W": _whole(r.W), "hist": _whole(r.hist), "bytes": int(r.out_bytes),
                "scans": np.array([[s[f] for f in whole] for s in r.scans], dtype=np.int64),
                "components": int(r.finish["components"]), "largest": int(r.finish["largest"])}
    if kind == "count":
        _load(st)
        hist, reads, total, counts = st["ctx"].count(want_counts=True)
        return {"hist": _whole(hist), "reads": _whole(reads), "total": int(total), "counts": counts.view(np.int32)}
    if kind == "noalloc":
        C, total = int(c["chunks"]), ctypes.c_uint64(0)
        p64 = ctypes.POINTER(ctypes.c_uint64)
        rc = mp.lib().mp_count_chunks_noalloc(
            torch.cuda.current_device(), int(c["k"]), 1 if c["min3"] else 0, st["fq"].data_ptr(), st["nbytes"],
            st["cofs"].ctypes.data_as(p64), C, st["counts"].ctypes.data, st["reads"].ctypes.data_as(p64),
            ctypes.byref(total))
        if rc:
            raise mp.MPError(rc, "mp_count_chunks_noalloc")
        return {"reads": _whole(st["reads"]), "total": int(total.value), "counts": st["counts"].view(np.int32)}
    if kind == "batch":
        ctx = st["ctx"]
        ctx.batch_load_device(st["fq"].data_ptr(), int(st["ofs"][-1]), st["ofs"])
        res, scan, fin = ctx.batch_partition()
        nb = ctx.batch_write(None)
        return {"parent": np.concatenate([ctx.batch_parent(i) for i in range(len(res))]).view(np.int32),
                "W": np.stack([_whole(r["W"]) for r in res]), "bytes": nb,
                "samples": np.array([[r[f] for f in ("reads", "tuples", "components", "largest")] for r in res],
                                    dtype=np.int64),
                "scan": np.array([scan.tuples, scan.bad_labels, scan.zeroed_runs, scan.evaluated_runs],
                                 dtype=np.int64)}
    srv = st["srv"]
    jobs = [srv.submit(b, want_parent=True) for b in st["jobs"]]
    got = [srv.wait(j, want_parent=True) for j in jobs]
    return {"parent": np.concatenate([p for _, p in got]).view(np.int32), "W": np.stack([_whole(d["W"]) for d, _ in got]),
            "jobs": np.array([[d[f] for f in ("reads", "tuples", "components", "largest")] for d, _ in got],
                             dtype=np.int64)}


def work(case):
    """FASTQ bytes in; the partitioned bytes (as many as came in, at the least) and one label per read out, or the
    counts.  No floating-point operation is needed."""
    c = dict(case)
    record = 16 + c["len_min"] + c["len_max"]
    kind = c["kind"]
    if kind in ("batch", "serve"):
        n = c["samples"] if kind == "batch" else c["jobs"]
        lo, hi = c["reads_min"], c["reads_max"]
        reads = n * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        return {"bytes": reads * (record * (2 if kind == "batch" else 1) + 4), "flops": 0}
    if kind == "partition":
        return {"bytes": c["reads"] * (record * (2 if c["write"] else 1) + 8), "flops": 0}
    return {"bytes": c["reads"] * record + 4.0 * c["chunks"] * (mp.NBUCKETS + 2), "flops": 0}


def exact(case, seed):
    return None
