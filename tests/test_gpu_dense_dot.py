"""Dense raw pass by two-element dot products: sums bit-equal to the oracle's at
remainders of the 16-frame groups and of the load ring, detectors that end
inside a wave, odd frame alignments, dark scales, totals that flush the 32-bit
lag sums, and pixels too bright for 16-bit groups (left to the FP64 kernel, seen
ahead or in passing)."""
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


def check_dense(xmt, orc, W, H, dpl, F, dq, sq, dark, counts):
    """Sums of dense frames (after the dark frames, no threshold) against the oracle's."""
    imm = synth.imm_bytes_dense(np.concatenate([dark, counts]).astype(np.uint16), W, H)
    plan = xmt.Plan(W, H, F, dpl, dq, sq, dark_frames=len(dark))
    plan.ingest_imm(imm)
    plan.execute()
    g, a, b = plan.sums()
    plan.close()
    r = orc.run_exact(imm, dq, sq, F, dpl, darks=len(dark))
    assert np.array_equal(a, r["IP"]) and np.array_equal(b, r["IF"])
    assert np.array_equal(g, r["G2"])


@pytest.mark.parametrize("dpl", [4, 8])
@pytest.mark.parametrize("darks", [0, 1, 2, 3, 11])
def test_groups_at_the_limit(xmt, orc, dpl, darks):
    """Groups of 16 frames whose (scaled) counts sum to what a wave of the dot
    kernel takes and just beyond, in one frame or over all of them, waves of
    every kind side by side."""
    W, H, F = 128, 5, 203
    n = max(darks, 1)
    limit = 64500 // 2 if darks == 1 else 64500
    ones = np.ones((H, W), np.int32)
    counts = np.zeros((F, W * H), np.int64)
    rng = np.random.default_rng(dpl + darks)
    for w in range(W * H // 64):
        px = slice(64 * w, 64 * w + 64)
        top = limit // n + (1 if w in (3, 8) else 0)         # waves 3 and 8 pass the limit
        k = w % 4
        if k == 0:      # one frame of every group, at any place in it
            counts[rng.integers(0, 16) + 16 * np.arange(F // 16), 64 * w + 5] = top
        elif k == 1:    # over the group
            counts[:, px] = top // 16
        elif k == 2:    # a few frames a group, every pixel its own
            for j in range(64):
                f = rng.choice(16, 4, replace=False)
                for g0 in range(0, F - 15, 16):
                    counts[g0 + f, 64 * w + j] = top // 4
        else:           # the largest raw value once, late
            counts[:, px] = rng.integers(0, 50, (F, 64))
            counts[F - 20, 64 * w + 7] = 65535 if w == 7 else top
    dark = rng.integers(0, 3, (darks, W * H))
    raw = np.minimum(counts + (dark.sum(0) // n if darks else 0), 65535)
    print(f"groups at the limit dpl={dpl} darks={darks}", flush=True)
    check_dense(xmt, orc, W, H, dpl, F, ones, ones, dark, raw)


@pytest.mark.parametrize("dpl", [4, 8])
@pytest.mark.parametrize("W,H,bright,late", [
    (128, 5, 0, 1), (128, 5, 1, 0), (128, 5, 10, 0),          # one wave leaves all to the FP64 kernel
    (384, 352, 3, 2), (384, 352, 527, 0), (384, 352, 1400, 5),  # 2112 waves: a quarter or five eighths do
])
def test_bright_waves_seen_ahead(xmt, orc, dpl, W, H, bright, late):
    """Waves bright throughout, which the look across the run finds, and ones
    bright in a single group, which it does not."""
    F = 1040
    npd, nw = W * H, W * H // 64
    rng = np.random.default_rng(W + bright + dpl)
    pix = np.arange(npd)
    q = (pix % 64 == 9).reshape(H, W).astype(np.int32)          # one mapped pixel a wave
    order = rng.permutation(nw)
    lam = np.full(npd, 3.0)
    lam[64 * order[:bright] + 9] = 5000.0
    counts = np.zeros((F, npd), np.uint16)
    on = pix[pix % 64 == 9]
    counts[:, on] = np.minimum(rng.poisson(lam[on], (F, len(on))), 65535)
    for w in order[bright:bright + late]:
        counts[1000, 64 * w + 9] = 65000
    print(f"bright waves {W}x{H} dpl={dpl} bright={bright} late={late}", flush=True)
    check_dense(xmt, orc, W, H, dpl, F, q, q, np.zeros((0, npd)), counts)


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
