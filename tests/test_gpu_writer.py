"""The writer's files against records sorted by file in Python, where its tiles
(256 reads, cut at the groups' ends) can go wrong: fewer reads than a wave,
tiles one record short or long, groups of a few reads, every group its own
tile, one file that takes nearly all, and batches."""
import glob
import os

import numpy as np
import pytest

import metapart_amd as mp

PARTS = 16


def _files(d):
    return {os.path.relpath(f, d): open(f, "rb").read() for f in glob.glob(d + "/**/*.fastq", recursive=True)}


def _records(buf):
    ends = np.flatnonzero(buf == 10)[3::4] + 1
    return [buf[a:b].tobytes() for a, b in zip(np.concatenate([[0], ends[:-1]]), ends)]


def _part(W, x):
    return next((p for p in range(PARTS - 1) if x < W[p + 1]), PARTS - 1)


def _reads(n, seed, deep):
    return mp.synth(0, n_reads=n, seed=seed, read_len_min=30, read_len_max=90,
                    **(dict(n_genomes=1, genome_len_min=3000, genome_len_max=3000) if deep else {}))


@pytest.mark.gpu
@pytest.mark.parametrize("n,C,T,deep", [(40, 1, 1, False), (254, 1, 1, False), (256, 2, 2, False), (258, 1, 1, True),
                                        (516, 2, 2, True), (1500, 60, 60, False), (5000, 6, 3, True),
                                        (70000, 16, 4, False)])
def test_files_of_singles(n, C, T, deep, tmp_path):
    print("gpu writer", n, C, T, flush=True)
    (tmp_path / "Rank0").mkdir()
    src = _reads(n, 70 + C, deep)
    buf = np.array(src.view(), copy=True)
    with mp.Context(k=27) as ctx:
        ctx.load(buf, mp.index_buffer(buf, C))
        r = mp.partition(ctx, S=1, T=1, want_parent=True, build_output=False)
        ids = ctx.first_ids()
        total = ctx.write_partitions(str(tmp_path), T, r.W)
    recs = _records(buf)
    want = {"Rank0/FromTid%d_ToRank%d.paired.fastq" % (t, p): [] for t in range(T) for p in range(PARTS)}
    for c in range(C):
        for i in range(int(ids[c]), int(ids[c + 1])):
            want["Rank0/FromTid%d_ToRank%d.paired.fastq" % (c // (C // T), _part(r.W, int(r.parent[i])))].append(recs[i])
    assert total == buf.nbytes
    assert _files(str(tmp_path)) == {k: b"".join(v) for k, v in want.items()}


@pytest.mark.gpu
def test_files_of_a_batch(tmp_path):
    print("gpu writer batch", flush=True)
    sizes = [40, 256, 258, 2, 900, 6000]
    srcs = [_reads(n, 90 + n, n > 800) for n in sizes]
    bufs = [np.array(s.view(), copy=True) for s in srcs]
    with mp.Context(k=27) as ctx:
        ctx.batch_load(bufs)
        res, _, _ = ctx.batch_partition()
        parents = [ctx.batch_parent(i) for i in range(len(bufs))]
        ctx.batch_write(str(tmp_path))
    want = {}
    for i, (buf, res_i, par) in enumerate(zip(bufs, res, parents)):
        files = [[] for _ in range(PARTS)]
        for j, rec in enumerate(_records(buf)):
            files[_part(res_i["W"], int(par[j]))].append(rec)
        for p in range(PARTS):
            want["sample%d/Rank0/FromTid0_ToRank%d.paired.fastq" % (i, p)] = b"".join(files[p])
    assert _files(str(tmp_path)) == want
