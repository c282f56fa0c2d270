"""One plan through several ingests: what an earlier one left (its buffers, work
that is still queued) does not reach the sums of a later one."""
import numpy as np
import pytest

import cases
import synth

pytestmark = pytest.mark.gpu


def rows_of(counts):
    """Pixel-major rows (row_off, frame, count) of counts [F, W * H]."""
    off = np.concatenate([[0], np.cumsum((counts > 0).sum(0))]).astype(np.int64)
    px, fr = np.nonzero(counts.T)
    return off, fr.astype(np.int32), counts[fr, px].astype(np.uint32)


def check(plan, ref):
    g, a, b = plan.sums()
    assert np.array_equal(g, ref["G2"]) and np.array_equal(a, ref["IP"]) and np.array_equal(b, ref["IF"])


@pytest.mark.parametrize("first", ["rows", "imm"])
def test_rows_then_fewer_imm_events(xmt, orc, first):
    """Rows handed in size the event buffer, not the transpose's: a compressed
    image of fewer events, and of more than any image before, follows."""
    big = cases.sparse_case(mu=0.6, seed=11)
    small = cases.sparse_case(mu=0.05, seed=12)
    mid = cases.sparse_case(mu=0.3, seed=13)
    plan = xmt.Plan(big["W"], big["H"], big["F"], big["dpl"], big["dq"], big["sq"])
    if first == "imm":     # a transpose buffer too small for what follows
        plan.ingest_imm(small["imm"])
        plan.execute()
        check(plan, orc.run_exact(small["imm"], small["dq"], small["sq"], small["F"], small["dpl"]))
    for c in (mid, small):
        print("rows, then image", first, int((c["counts"] > 0).sum()), flush=True)
        plan.ingest_rows(*rows_of(big["counts"]))
        plan.execute()
        check(plan, orc.run_exact(big["imm"], big["dq"], big["sq"], big["F"], big["dpl"]))
        plan.ingest_imm(c["imm"])
        plan.execute()
        check(plan, orc.run_exact(c["imm"], c["dq"], c["sq"], c["F"], c["dpl"]))
    plan.close()


def test_refused_frames_leave_the_data(xmt, orc):
    """Frames refused for a value leave the plan's data as it was, also where
    they would have needed a larger buffer."""
    c = cases.sparse_case(mu=0.05, seed=21)
    plan = xmt.Plan(c["W"], c["H"], c["F"], c["dpl"], c["dq"], c["sq"])
    frames = np.ones((c["F"], c["W"] * c["H"]), np.uint32)
    frames[-1, -1] = 65536
    with pytest.raises(xmt.XpcsError, match="UNSUPPORTED"):
        plan.ingest_frames(frames)
    with pytest.raises(xmt.XpcsError, match="STATE"):
        plan.execute()
    plan.ingest_imm(c["imm"])
    with pytest.raises(xmt.XpcsError, match="UNSUPPORTED"):
        plan.ingest_frames(frames)
    plan.execute()
    check(plan, orc.run_exact(c["imm"], c["dq"], c["sq"], c["F"], c["dpl"]))
    frames[-1, -1] = 65535
    plan.ingest_frames(frames)
    plan.execute()
    want = frames.astype(np.uint16)
    check(plan, orc.run_exact(synth.imm_bytes_dense(want, c["W"], c["H"]), c["dq"], c["sq"], c["F"], c["dpl"]))
    plan.close()


def busy_stream():
    """A torch stream with a tenth of a second of work queued."""
    import torch
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        torch.cuda._sleep(200_000_000)
    return s


INGESTS = {
    "imm": lambda xmt, plan, c, W, H: plan.ingest_imm(synth.imm_bytes_sparse(c, W, H)),
    "dense": lambda xmt, plan, c, W, H: plan.ingest_imm(synth.imm_bytes_dense(c, W, H)),
    "frames": lambda xmt, plan, c, W, H: plan.ingest_frames(c),
    "rows": lambda xmt, plan, c, W, H: plan.ingest_rows(*rows_of(c)),
    "ufxc": lambda xmt, plan, c, W, H: plan.ingest_packed(synth.ufxc_words(c, W, H), xmt.FMT_UFXC),
    "events": lambda xmt, plan, c, W, H: plan.ingest_events(
        np.nonzero(c)[1].astype(np.int32), c[np.nonzero(c)].astype(np.uint16),
        np.concatenate([[0], np.cumsum((c > 0).sum(1))]).astype(np.int64)),
}


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("kind", sorted(INGESTS))
def test_ingest_waits_for_a_callers_stream(xmt, orc, kind, batch):
    """The plan's previous data is still to be read by work on another stream
    when the next data is handed in: the ingest waits for it, and the sums are
    the new data's."""
    import torch
    W, H, F = 32, 24, 150
    dq, sq = synth.annular_qmaps(W, H, 6, 3)
    data = [np.minimum(synth.ou_counts(W, H, F, 0.2, 8.0, seed=k), 3).astype(np.uint16) for k in (1, 2, 3)]
    plan = xmt.Plan(W, H, F, 4, dq, sq)
    ingest = INGESTS[kind]
    ingest(xmt, plan, data[0], W, H)
    plan.execute()
    plan.sums()
    jobs = xmt.Batch()
    if batch:
        jobs.add(plan)
        jobs.execute()
        jobs.synchronize()
    for c in data[1:]:
        print("ingest after work on another stream:", kind, batch, flush=True)
        s = busy_stream()
        (jobs if batch else plan).execute(stream=s.cuda_stream)
        done = s.record_event()
        assert not done.query()
        ingest(xmt, plan, c, W, H)
        assert done.query()
        plan.execute()
        check(plan, orc.run_exact(synth.imm_bytes_sparse(c, W, H), dq, sq, F, 4))
    torch.cuda.synchronize()
    jobs.close()
    plan.close()
