"""The pair step against the sequential loop, on reads whose components are known
by construction (reads of one contig are equal, contigs share no k-mer): pair
numbers in order along chains of components (what the rounds on the device leave
to the host), against them and in no order, stars around large components, and
components that pass 1000 reads on the way."""
import numpy as np
import pytest

import metapart_amd as mp

GATE = 1000
BIG = 120000  # pairs: enough for the rounds on the device


def _loop(contig):
    """labels after the pair step: the reference's loop over (2j, 2j + 1)"""
    n = len(contig)
    comp = {}
    for i, c in enumerate(contig):
        comp.setdefault(int(c), []).append(i)
    lab = {c: (max(m), len(m)) for c, m in comp.items()}
    up = {c: c for c in comp}

    def find(x):
        while up[x] != x:
            up[x] = up[up[x]]
            x = up[x]
        return x
    for j in range(n // 2):
        a, b = find(int(contig[2 * j])), find(int(contig[2 * j + 1]))
        if a == b or (lab[a][1] > GATE and lab[b][1] > GATE):
            continue
        up[b] = a
        lab[a] = (max(lab[a][0], lab[b][0]), lab[a][1] + lab[b][1])
    return np.array([lab[find(int(c))][0] for c in contig], dtype=np.uint64)


def _chain(m, order, seed):
    p = np.stack([np.arange(m), np.arange(1, m + 1)], axis=1)
    if order == "descending":
        p = p[::-1]
    if order == "shuffled":
        p = np.random.default_rng(seed).permutation(p)
    return p


def _pairs(kind):
    rng = np.random.default_rng(9)
    if kind.startswith("chain"):
        return _chain(BIG, kind[6:], 1)
    if kind == "two_chains":  # both pass 1000 reads; cross pairs before, among and after
        m = BIG // 2
        a, b = _chain(m, "shuffled", 2), _chain(m, "shuffled", 3) + m + 1
        cross = np.stack([rng.integers(0, m, 15000), m + 1 + rng.integers(0, m, 15000)], axis=1)
        p = np.concatenate([a, b, cross])
        return p[rng.permutation(len(p))]
    if kind == "stars":  # four large contigs, thousands of small ones between them
        hub = np.repeat(np.arange(4), 600)[:, None].repeat(2, axis=1)
        spokes = np.stack([rng.integers(0, 4, BIG), 4 + rng.integers(0, 70000, BIG)], axis=1)
        flip = rng.random(len(spokes)) < 0.5
        spokes[flip] = spokes[flip][:, ::-1]
        return np.concatenate([hub, spokes])[rng.permutation(2400 + BIG)]
    if kind == "parallel":  # few contigs, most of them joined by several pairs
        return np.minimum(rng.geometric(0.0002, (BIG, 2)), 40000)
    if kind == "wide":
        return rng.integers(0, 100000, (BIG + 20000, 2))
    if kind == "few":  # too few for the rounds
        return rng.integers(0, 2500, (3000, 2))
    raise ValueError(kind)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["chain_ascending", "chain_descending", "chain_shuffled", "two_chains", "stars",
                                  "parallel", "wide", "few"])
def test_pair_step_equals_the_loop(kind):
    print("gpu pair step", kind, flush=True)
    contig = _pairs(kind).reshape(-1)
    letters = np.frombuffer(b"ACGT", np.uint8)
    seqs = [s.tobytes().decode() for s in np.random.default_rng(4).choice(letters, (int(contig.max()) + 1, 44))]
    text = "".join("@r%d\n%s\n+\n%s\n" % (i, seqs[c], "I" * 44) for i, c in enumerate(contig))
    buf = np.frombuffer(text.encode(), dtype=np.uint8).copy()
    with mp.Context(k=27) as ctx:
        ctx.load(buf, mp.index_buffer(buf, 4))
        r = mp.partition(ctx, S=1, T=1, want_parent=True, build_output=False)
    want = _loop(contig)
    assert np.array_equal(np.asarray(r.parent), want)
