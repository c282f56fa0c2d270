"""Row kernels (a group of lanes per pixel row): sums bit-equal to the oracle's
at the edges of the row classes, with repeated frames, with frames left over
at every level and with long frame counts.  Many of the rows hold counts above
65535, so the kernels of k_multitau.hip take them all; the same lengths and
orders on the row kernels, the totals that fit their 16 bits and the frame
counts that fit their keys are in test_gpu_wide_rows.py."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dpl,F", [(4, 40), (4, 1023), (8, 2500), (8, 10007), (4, 65000), (8, 65530)])
@pytest.mark.parametrize("order", ["sorted", "local", "shuffled"])
def test_row_classes(xmt, orc, dpl, F, order):
    rng = np.random.default_rng(1000 * dpl + F)
    W = H = 14
    npd = W * H
    dq, sq = synth.annular_qmaps(W, H, 4, 2)
    edges = [0, 1, 2, 7, 8, 9, 31, 63, 64, 65, 66, 127, 128, 129, 130, 500, 512, 513, 514, 1023, 1024, 1025, 1300]
    lens = rng.choice(edges, npd)
    frames, counts = [], []
    for j, n in enumerate(lens):
        # bursts, spread rows, and rows with repeated frames
        span = F if j % 3 else max(F // 7, 1)
        f = np.sort(rng.integers(0, span, n)) + (rng.integers(0, F - span + 1))
        c = rng.integers(1, 4, n).astype(np.int64)
        if n and j % 5 == 0:       # totals of 65534 .. 65537 and far beyond
            c[:] = 0
            c[rng.integers(0, n)] = [65534, 65535, 65536, 65537, 4000000][(j // 5) % 5]
            if j % 2 and n > 1:
                k = rng.integers(0, n)
                c[k] += c.max() // 2
        if order == "local":
            for a in range(0, n, 6):
                s = rng.permutation(min(6, n - a)) + a
                f[a:a + 6], c[a:a + 6] = f[s], c[s]
        elif order == "shuffled":
            s = rng.permutation(n)
            f, c = f[s], c[s]
        frames.append(f.astype(np.int32))
        counts.append(c.astype(np.uint32))
    roff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    print(f"rows dpl={dpl} F={F} order={order}", flush=True)
    plan = xmt.Plan(W, H, F, dpl, dq, sq)
    plan.ingest_rows(roff, np.concatenate(frames), np.concatenate(counts))
    plan.execute()
    g, a, b = plan.sums()
    total = plan.side()["pixel_sum"]
    plan.close()
    ordr = orc.build_qmap(dq, sq)["order"]
    # the oracle takes rows in frame order
    srt = [np.argsort(frames[j], kind="stable") for j in ordr]
    csr = dict(off=np.concatenate([[0], np.cumsum(lens[ordr])]).astype(np.int64),
               frame=np.concatenate([frames[j][s] for j, s in zip(ordr, srt)]),
               cnt=np.concatenate([counts[j][s] for j, s in zip(ordr, srt)]).astype(np.int64))
    lev, tau = orc.schedule(F, dpl)
    G2, IP, IF = orc.multitau_exact(csr, F, lev, tau)
    assert np.array_equal(a, IP) and np.array_equal(b, IF)
    assert np.array_equal(g, G2)
    want = np.array([counts[j].astype(np.float64).sum() / F for j in ordr])
    np.testing.assert_allclose(total[ordr], want, rtol=1e-6)
