"""3-minimizer scans of reads a few bases longer than k, where a read's windows
are one or two k-mers wide and it yields the most tuples a read can (five at
k + 5 bases), against the oracle."""
import pytest

from test_gpu_stages import _check_stages

CASES = [("min3_short_k27", dict(n_reads=8000, seed=141, read_len_min=27, read_len_max=36), 4, 27, 1, 1, True, False, 0),
         ("min3_k_plus_5", dict(n_reads=4000, seed=142, read_len=36), 4, 31, 1, 1, True, False, 0),
         ("min3_odd_workgroup", dict(n_reads=514, seed=143, read_len_min=25, read_len_max=60, n_rate=0.01), 2, 20, 1, 2, True,
          False, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_short_reads_match_oracle(case, tmp_path):
    print("gpu min3 short reads", case[0], flush=True)
    _check_stages(case, tmp_path)
