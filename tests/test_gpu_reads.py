"""Large results read while other threads use the library, and with another
device current."""
import threading
import time

import numpy as np
import pytest

import cases
import synth

pytestmark = pytest.mark.gpu


def executed(xmt, W, F, seed):
    """A plan whose G2 is several megabytes, and that G2."""
    dq, sq = synth.annular_qmaps(W, W, 6, 3)
    rng = np.random.default_rng(seed)
    counts = (rng.random((F, W * W)) < 0.02).astype(np.uint16) * rng.integers(1, 4, (F, W * W)).astype(np.uint16)
    plan = xmt.Plan(W, W, F, 4, dq, sq)
    plan.ingest_imm(synth.imm_bytes_sparse(counts, W, W))
    plan.execute()
    return plan, plan.sums()[0]


def read_into(xmt, plan, out):
    xmt.check(xmt.lib().xpcs_mt_read_sums_i64(plan._h, xmt._p(out), None, None))


def test_reads_during_an_ingest(xmt):
    """A read of megabytes does not wait for another thread's upload."""
    reader, G2 = executed(xmt, 256, 200, 1)
    assert G2.nbytes > 8 << 20
    W, F = 512, 6000          # 3 GB of frames, more than 50 ms of upload
    ones = np.ones((W, W), np.int32)
    big = xmt.Plan(W, W, F, 4, ones, ones)
    frames = np.zeros((F, W * W), np.uint16)
    out = np.empty_like(G2)
    read_into(xmt, reader, out)                # buffers made, pages touched
    span = []

    def ingest():
        t = time.perf_counter()
        big.ingest_frames(frames)
        span.extend([t, time.perf_counter()])
    th = threading.Thread(target=ingest)
    reads = []
    th.start()
    while th.is_alive():
        out[:] = -1
        t = time.perf_counter()
        read_into(xmt, reader, out)
        reads.append((t, time.perf_counter()))
        assert np.array_equal(out, G2)
    th.join()
    inside = [r for r in reads if r[0] > span[0] and r[1] < span[1]]
    print(f"upload {1e3 * (span[1] - span[0]):.0f} ms, {len(inside)} reads within", flush=True)
    big.close()
    reader.close()
    assert len(inside) >= 3


def test_reads_of_several_threads(xmt):
    plans = [executed(xmt, 192 + 16 * k, 150, k) for k in range(4)]
    bad = []

    def work(plan, G2):
        out = np.empty_like(G2)
        for _ in range(10):
            out[:] = -1
            read_into(xmt, plan, out)
            if not np.array_equal(out, G2):
                bad.append(plan)
    ths = [threading.Thread(target=work, args=p) for p in plans]
    for th in ths:
        th.start()
    for th in ths:
        th.join()
    for p, _ in plans:
        p.close()
    assert not bad


def test_read_with_another_device_current(xmt):
    import torch
    if torch.cuda.device_count() < 2:
        pytest.skip("one device")
    with torch.cuda.device(0):
        plan, G2 = executed(xmt, 256, 200, 2)
        c = cases.sparse_case(W=64, H=64, F=1200, mu=0.1)
        tt = xmt.Plan(64, 64, 1200, 4, c["dq"], c["sq"])
        tt.ingest_imm(c["imm"])
        want = tt.twotime([1])["c2t"][0]
    with torch.cuda.device(1):
        out = np.empty_like(G2)
        read_into(xmt, plan, out)
        c2t = np.empty_like(want)
        xmt.check(xmt.lib().xpcs_mt_read_twotime(tt._h, 0, xmt._p(c2t)))
        assert np.array_equal(out, G2) and np.array_equal(c2t, want)
    plan.close()
    tt.close()
