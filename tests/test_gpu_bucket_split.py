"""Transposes whose buckets hold more events than the row placement stages:
halved to 128 rows, beyond that in batches; exact against the oracle."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,F,mu,shift", [
    (32, 32, 2000, 0.1, 8),     # 51k events a bucket of 256 rows: stays
    (33, 31, 3200, 0.1, 0),     # 80k: 128 rows, the last bucket ragged
    (32, 32, 3000, 0.6, 0),     # 300k, 150k after halving: batches of 128-row buckets
])
def test_halved_buckets(xmt, orc, W, H, F, mu, shift):
    c = cases.sparse_case(W=W, H=H, F=F, dpl=4, mu=mu, tau_c=12.0, seed=41 + F)
    print("buckets", W, H, F, mu, flush=True)
    plan = xmt.Plan(W, H, F, 4, c["dq"], c["sq"])
    plan.ingest_imm(c["imm"])
    plan.execute()
    assert plan.get_tuning()["tr_bucket_shift"] == shift
    r = orc.run_exact(c["imm"], c["dq"], c["sq"], F, 4)
    G2, IP, IF = plan.sums()
    assert np.array_equal(IP, r["IP"]) and np.array_equal(IF, r["IF"]) and np.array_equal(G2, r["G2"])
    plan.close()
