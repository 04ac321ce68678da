"""The union of listed runs in two parts (over a million reads, many live labels
a read): runs that go on across the cut, against the radix path."""
import numpy as np
import pytest

import metapart_amd as mp


@pytest.mark.gpu
@pytest.mark.parametrize("genomes,length,sigma", [(1, 500000, 0.0), (40, 40000, 1.5)])
def test_two_parts_equal_radix(genomes, length, sigma):
    print("gpu union in two parts", genomes, flush=True)
    buf = mp.synth(0, n_reads=1100000, seed=31, read_len=70, n_genomes=genomes, genome_len_min=length, genome_len_max=length,
                   abund_sigma=sigma, err_rate=0.001)
    got = []
    for kw in ({}, dict(sort_digit_bits=7)):  # a digit width asks for the radix sort
        with mp.Context(k=27, **kw) as ctx:
            ctx.load(buf, mp.index_buffer(buf, 2))
            r = mp.partition(ctx, S=1, T=1, want_parent=True, build_output=False)
            got.append((r.parent, r.W, [s["bad_labels"] for s in r.scans], r.scans[0]["ms_sort_gen"] == 0))
    assert got[0][3] and not got[1][3]
    assert 16 * len(got[0][0]) <= 1100000 * 44 * (1 - got[0][2][0] / len(got[0][0]))  # the rule's depth
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
