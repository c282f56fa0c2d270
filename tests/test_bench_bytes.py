"""Algorithmic bytes that the benchmark charges the sparse kernels."""
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent.parent))


def test_halved_buckets_have_128_rows():
    """A bucket shift of 0 in a reported tuning is the automatic choice of 2^7."""
    import bench
    px = np.array([1, 2, 3, 4, 5, 0])
    args = dict(T=30, E_raw=1000, nsel=100, nrows=100_000, n_mapped=80_000, px=px, ev=10 * px)
    got = bench.sparse_kernel_bytes(tuning=dict(tr_bucket_shift=0, tr_chunk_frames=2), **args)
    assert got == bench.sparse_kernel_bytes(tuning=dict(tr_bucket_shift=7, tr_chunk_frames=2), **args)
    # histogram in and segment offsets out: 782 buckets, 50 chunks
    assert got["k_tr_scan"] == 4 * 782 * 50 + 8 * (782 * 50 + 1)
