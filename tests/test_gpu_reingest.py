"""One plan through several ingests: what an earlier one left (its buffers, work
that is still queued) does not reach the sums of a later one."""
import numpy as np
import pytest

import cases

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
