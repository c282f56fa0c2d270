"""Dense raw pass by two-element dot products: sums bit-equal to the oracle's at
remainders of the 16-frame groups and of the load ring, detectors that end
inside a wave, odd frame alignments, dark scales, totals that flush the 32-bit
lag sums, and pixels too bright for 16-bit groups (left to the FP64 kernel)."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(15, 13), (24, 24), (101, 3)])
@pytest.mark.parametrize("dpl,F", [(4, 37), (4, 200), (8, 333), (8, 1024), (4, 1007)])
@pytest.mark.parametrize("darks,scale", [(0, 2), (2, 5), (3, 400), (1, 9000), (0, 60000)])
def test_dense_dot_sums(xmt, orc, W, H, dpl, F, darks, scale):
    rng = np.random.default_rng(W * 7 + F + scale)
    npd = W * H
    yy, xx = np.mgrid[0:H, 0:W]
    sq = (1 + (xx + yy) % 4).astype(np.int32)
    sq[(xx * 7 + yy * 3) % 11 == 0] = 0
    dq = np.where(sq > 0, 1 + (sq - 1) // 2, 0).astype(np.int32)
    lam = scale * rng.exponential(1.0, (F, npd)) * np.where(rng.random(npd) < 0.1, 0.02, 1.0)
    counts = np.minimum(rng.poisson(np.minimum(lam, 6.0e4)), 65000).astype(np.uint16)
    kw = {}
    if darks:
        dark = rng.poisson(3.0, (darks, npd)).astype(np.uint16)
        counts = np.minimum(counts.astype(np.int64) + dark[0], 65535).astype(np.uint16)
        raw = np.concatenate([dark, counts])
        kw = dict(darks=darks, lld=1.5, sigma=1.0)
    else:
        raw = counts
    imm = synth.imm_bytes_dense(raw, W, H)
    print(f"dense dot {W}x{H} dpl={dpl} F={F} darks={darks} scale={scale}", flush=True)
    plan = xmt.Plan(W, H, F, dpl, dq, sq, dark_frames=darks, lld=kw.get("lld", 0.0), sigma=kw.get("sigma", 0.0))
    plan.ingest_imm(imm)
    plan.execute()
    g, a, b = plan.sums()
    plan.close()
    r = orc.run_exact(imm, dq, sq, F, dpl, **kw)
    assert np.array_equal(a, r["IP"]) and np.array_equal(b, r["IF"])
    assert np.array_equal(g, r["G2"])


def test_buffers_of_a_short_run(xmt):
    """A short run on a large detector holds its boundary sums once, beside the
    first series."""
    torch = pytest.importorskip("torch")
    W, F, dpl = 1024, 64, 4
    ones = np.ones((W, W), np.int32)
    frames = np.ones((F, W * W), np.uint16)
    small = xmt.Plan(64, 64, F, dpl, ones[:64, :64], ones[:64, :64])   # the kernels' own memory first
    small.ingest_frames(frames[:, :64 * 64])
    small.execute()
    small.sums()
    plan = xmt.Plan(W, W, F, dpl, ones, ones)
    plan.ingest_frames(frames)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan.execute()
    plan.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    levels, taus = xmt.delays_per_level(F, dpl)
    bounds = set()
    for L, tau in zip(levels, taus):
        lf, t = F >> L, int(tau) >> L
        bounds |= {(lf - t) << L, t << L, lf << L}
    need = 4 * W * W * (len(bounds) + (F >> 4))
    print(f"buffers {used >> 20} MiB for {need >> 20}", flush=True)
    g, a, b = plan.sums()
    plan.close()
    small.close()
    assert used < 1.25 * need
    n = np.array([(F >> L) - (int(t) >> L) for L, t in zip(levels, taus)])
    assert (a[0] == n << levels).all() and (a == a[0]).all() and (b == a[0]).all()
    assert (g == (n << levels) << levels).all()
