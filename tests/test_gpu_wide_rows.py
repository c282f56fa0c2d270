"""Row kernels with totals on both sides of the 65535 that 16 bits hold: sums
bit-equal to the oracle's at the edges of the length classes, of the totals and
of the frame counts, narrow and wide rows mixed at every density, and rows with
counts that do not fit 16 bits."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 7, 8, 9, 31, 63, 64, 65, 66, 127, 128, 129, 130, 500, 512, 513, 514, 1023, 1024, 1025, 1300]


def check_rows(xmt, orc, W, H, F, dpl, frames, counts, row_kernels, deep=0):
    """Sums of pixel-major rows against the oracle's; row_kernels: the plan takes k_mt_rows."""
    dq, sq = synth.annular_qmaps(W, H, 4, 2)
    lens = np.array([len(f) for f in frames])
    plan = xmt.Plan(W, H, F, dpl, dq, sq)
    plan.ingest_rows(np.concatenate([[0], np.cumsum(lens)]).astype(np.int64),
                     np.concatenate(frames).astype(np.int32), np.concatenate(counts).astype(np.uint32))
    plan.set_tuning(deep_frames=deep)
    # the path taken: the row kernels' series has the level's frames, the other
    # kernels' whole 16 bytes of them, by default from 96 frames on
    info = plan.info()
    lf = F >> info.deep_level
    assert info.deep_stride == (lf if row_kernels else (lf + 3) & ~3)
    assert plan.get_tuning()["deep_frames"] == (deep if deep else 0 if row_kernels else 96)
    plan.execute()
    g, a, b = plan.sums()
    total = plan.side()["pixel_sum"]
    plan.close()
    order = orc.build_qmap(dq, sq)["order"]
    # the oracle takes rows in frame order
    srt = [np.argsort(frames[j], kind="stable") for j in order]
    csr = dict(off=np.concatenate([[0], np.cumsum(lens[order])]).astype(np.int64),
               frame=np.concatenate([frames[j][s] for j, s in zip(order, srt)]).astype(np.int32),
               cnt=np.concatenate([counts[j][s] for j, s in zip(order, srt)]).astype(np.int64))
    lev, tau = orc.schedule(F, dpl)
    G2, IP, IF = orc.multitau_exact(csr, F, lev, tau)
    assert np.array_equal(a, IP) and np.array_equal(b, IF)
    assert np.array_equal(g, G2)
    want = np.array([counts[j].astype(np.float64).sum() / F for j in order])
    np.testing.assert_allclose(total[order], want, rtol=1e-6)


def draw_rows(rng, npd, F, wide):
    """Rows of every class; a row is wide with probability `wide`: totals of
    65535 (narrow still), 65536 and far beyond, from several counts."""
    frames, counts = [], []
    for j, n in enumerate(rng.choice(EDGES, npd)):
        span = F if j % 3 else max(F // 7, 1)       # spread rows and bursts
        f = np.sort(rng.integers(0, span, n)) + rng.integers(0, F - span + 1)
        if j % 4 == 3:                              # events in the last frames
            f = np.minimum(f + F, F - 1 - rng.integers(0, min(F, 3), n))
        c = rng.integers(1, 4, n).astype(np.int64)
        if n > 1 and rng.random() < wide:
            k = j % 3
            if k < 2:
                c[-1] = 65535 + k - c[:-1].sum()    # 65535 and 65536
            else:
                c[:] = rng.integers(1, 65536, n)
                c[rng.integers(0, n, 2)] = 65535
        s = rng.permutation(n)
        frames.append(f[s].astype(np.int32))
        counts.append(c[s].astype(np.uint32))
    return frames, counts


@pytest.mark.parametrize("dpl,F", [(4, 40), (4, 1023), (8, 2500), (8, 10007), (4, 30011)])
@pytest.mark.parametrize("wide", [0.02, 0.4, 1.0])
def test_wide_rows(xmt, orc, dpl, F, wide):
    rng = np.random.default_rng([dpl, F, int(100 * wide)])
    print(f"wide rows dpl={dpl} F={F} wide={wide}", flush=True)
    check_rows(xmt, orc, 20, 17, F, dpl, *draw_rows(rng, 340, F, wide), True)


@pytest.mark.parametrize("dpl", [4, 8])
@pytest.mark.parametrize("F", [17, 32, 33, 96, 97, 192, 193, 768, 769, 1536, 1537, 3072, 3073])
def test_series_from_level_0(xmt, orc, dpl, F):
    """Frame counts around the limits below which a length class sums level 0
    from its series too, rows with many events a frame among them."""
    rng = np.random.default_rng([dpl, F])
    print(f"level 0 series dpl={dpl} F={F}", flush=True)
    check_rows(xmt, orc, 20, 17, F, dpl, *draw_rows(rng, 340, F, 0.3), True)


@pytest.mark.parametrize("dpl,F,deep,row_kernels", [
    (4, 63231, 0, True), (4, 63232, 0, False), (8, 61183, 0, True), (8, 61184, 0, False),
    (8, 65535 - 17 * 512, 96, True), (8, 65536 - 17 * 512, 96, False),
    (4, 65535 - 9 * 2048, 16, True), (4, 65536 - 9 * 2048, 16, False),
])
def test_frame_limit(xmt, orc, dpl, F, deep, row_kernels):
    """The largest frame count whose keys leave the padding key out of reach,
    and the next one, which the other kernels take; rows with events in the
    last frames among them."""
    rng = np.random.default_rng(F)
    print(f"frame limit dpl={dpl} F={F} deep_frames={deep}", flush=True)
    check_rows(xmt, orc, 20, 17, F, dpl, *draw_rows(rng, 340, F, 0.3), row_kernels, deep)


@pytest.mark.parametrize("order", ["sorted", "local", "shuffled"])
@pytest.mark.parametrize("dpl,F", [(4, 1023), (8, 10007)])
def test_narrow_rows_in_any_order(xmt, orc, dpl, F, order):
    rng = np.random.default_rng([dpl, F, len(order)])
    frames, counts = draw_rows(rng, 340, F, 0.0)
    for j, f in enumerate(frames):
        if order != "shuffled":
            f.sort()
        if order == "local":
            for a in range(0, len(f), 6):
                f[a:a + 6] = rng.permutation(f[a:a + 6])
    print(f"rows dpl={dpl} F={F} order={order}", flush=True)
    check_rows(xmt, orc, 20, 17, F, dpl, frames, counts, True)


@pytest.mark.parametrize("big", [1, 10, 11])
def test_counts_above_16_bits(xmt, orc, big):
    """Up to one row in 32 with such a count goes to a list, more to the kernels
    without 16-bit counts."""
    rng = np.random.default_rng(big)
    W, H, F = 20, 17, 5000
    frames, counts = draw_rows(rng, W * H, F, 0.3)
    dq, sq = synth.annular_qmaps(W, H, 4, 2)
    mapped = [j for j in np.flatnonzero(((dq > 0) & (sq > 0)).reshape(-1)) if 0 < len(frames[j]) <= 1024]
    limit = int(((dq > 0) & (sq > 0)).sum()) // 32
    n = big if big < 10 else limit + big - 10
    assert 1 < limit < len(mapped) - 1
    for j in rng.choice(mapped, n, replace=False):
        counts[j][rng.integers(0, len(counts[j]))] = 65536 + 1000 * (j % 3)
    print("big counts", n, limit, flush=True)
    check_rows(xmt, orc, W, H, F, 8, frames, counts, n <= limit)


def test_wide_rows_of_an_image(xmt, orc):
    """Compressed frames of large counts, all rows wide, against the oracle."""
    W, H, F = 64, 48, 900
    dq, sq = synth.annular_qmaps(W, H, 6, 3)
    counts = synth.ou_counts(W, H, F, 0.1, 8.0, seed=3).astype(np.int64)
    rng = np.random.default_rng(4)
    counts = np.where(counts > 0, np.minimum(counts * 1500 + rng.integers(0, 700, counts.shape), 65535), 0)
    imm = synth.imm_bytes_sparse(counts.astype(np.uint16), W, H)
    ref = orc.run_exact(imm, dq, sq, F, 8)
    plan = xmt.Plan(W, H, F, 8, dq, sq)
    plan.ingest_imm(imm)
    plan.execute()
    g, a, b = plan.sums()
    g2, _ = plan.g2()
    plan.close()
    assert np.array_equal(g, ref["G2"]) and np.array_equal(a, ref["IP"]) and np.array_equal(b, ref["IF"])
    np.testing.assert_allclose(g2, ref["g2"], rtol=1e-12)
