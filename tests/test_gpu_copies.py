"""Copies through the pinned buffers: uploads at the line from which they are
staged and at whole and odd numbers of buffers, counts and labels down, each
against the same data by a direct copy; and all of them without pinned memory."""
import os
import subprocess
import sys

import numpy as np
import pytest

import metapart_amd as mp

MB = 1 << 20


def _sized(view, nbytes):
    """whole records from the front of `view`, the first one's name stretched to make nbytes"""
    ends = np.flatnonzero(view[:nbytes - 4] == 10)[3::4]  # a record's fourth newline
    cut = int(ends[-1]) + 1
    first = int(np.flatnonzero(view[:1000] == 10)[0])
    out = np.empty(nbytes, np.uint8)
    pad = nbytes - cut
    out[:first] = view[:first]
    out[first:first + pad] = ord("x")
    out[first + pad:] = view[first:cut]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("nbytes", [32 * MB - 1, 32 * MB, 40 * MB, 40 * MB + 1])
def test_staged_upload_and_counts(nbytes):
    import torch
    print("gpu staged upload", nbytes, flush=True)
    src = mp.synth(0, n_reads=200000, seed=5, read_len=100)
    buf = _sized(src.view(), nbytes)
    assert len(buf) == nbytes
    dev = torch.from_numpy(buf).to("cuda")
    got = []
    for C in (1, 5):  # 4 MB of counts by a direct copy, 20 MB staged
        with mp.Context(k=27) as ctx:
            ctx.load(buf, mp.index_buffer(buf, C))
            got.append(ctx.count(want_counts=True)[3])
    with mp.Context(k=27) as ctx:
        ctx.load_device(dev.data_ptr(), nbytes, mp.index_buffer(buf, 1))
        want = ctx.count(want_counts=True)[3]
    assert want.sum() > 0
    assert np.array_equal(got[0], want)
    assert np.array_equal(got[1].sum(axis=0, dtype=np.uint64), want[0])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [MB - 2, MB, MB + 2, 3 * MB + 2])
def test_labels(n):
    print("gpu labels", n, flush=True)
    buf = mp.synth(0, n_reads=n, seed=6, read_len=30)
    with mp.Context(k=27) as ctx:
        ctx.load(buf, mp.index_buffer(buf, 1))
        mp.partition(ctx, S=1, T=1, build_output=False)
        got = ctx.parent()
    with mp.Context(k=27) as ctx:
        ctx.batch_load([buf])
        ctx.batch_partition()
        want = ctx.batch_parent(0)  # 32-bit, a direct copy
    assert len(got) == n and np.array_equal(got, want)


@pytest.mark.gpu
def test_copies_without_pinned_memory(tmp_path):
    # a process whose hipHostMalloc has no memory to give: uploads, counts and labels of the staged sizes go the
    # runtime's way
    print("gpu copies without pinned memory", flush=True)
    shim = tmp_path / "shim.c"
    shim.write_text("#include <stddef.h>\nint hipHostMalloc(void **p, size_t n, unsigned f) { *p = 0; return 2; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(shim)], check=True)
    prog = """if 1:
        import ctypes, sys
        ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
        import numpy as np
        import metapart_amd as mp
        buf = mp.synth(0, n_reads=%d, seed=6, read_len=30)
        assert buf.nbytes > 32 << 20
        with mp.Context(k=27) as ctx:
            ctx.load(buf, mp.index_buffer(buf, 5))
            counts = ctx.count(want_counts=True)[3]
            r = mp.partition(ctx, S=1, T=1, want_parent=True, build_output=False)
        np.savez(sys.argv[2], counts=counts.sum(axis=0, dtype=np.uint64), parent=r.parent)
    """ % (MB + 2)
    out = str(tmp_path / "out.npz")
    subprocess.run([sys.executable, "-c", prog, str(tmp_path / "shim.so"), out], check=True, timeout=100,
                   cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    got = np.load(out)
    buf = mp.synth(0, n_reads=MB + 2, seed=6, read_len=30)
    with mp.Context(k=27) as ctx:
        ctx.load(buf, mp.index_buffer(buf, 5))
        counts = ctx.count(want_counts=True)[3]
        r = mp.partition(ctx, S=1, T=1, want_parent=True, build_output=False)
    assert np.array_equal(got["counts"], counts.sum(axis=0, dtype=np.uint64)) and np.array_equal(got["parent"], r.parent)
