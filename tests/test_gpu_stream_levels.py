"""Stream kernels where their split can go wrong: more levels than a block has
waves, rows longer than one launch stores, pixel counts beside 64, pushes that
cross level boundaries at any phase.  Sums against numpy, whole numbers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def level_sums(x, taus, levels):
    """(G2, IP, IF) int64 [P, T] of counts x [F, P]; level L sums 2^L frames."""
    out, L, y = [], 0, x
    for tau, lev in zip(taus, levels):
        while L < lev:
            y = y[:len(y) // 2 * 2].reshape(-1, 2, y.shape[1]).sum(1)
            L += 1
        d = int(tau) >> L
        out.append(((y[:-d] * y[d:]).sum(0), y[:-d].sum(0), y[d:].sum(0)))
    return [np.stack(a, 1) for a in zip(*out)]


@pytest.mark.parametrize("W,H,F,dpl,piece,filled", [
    (7, 9, 70, 4, 1, 1.0),
    (13, 10, 700, 8, 65, 1.0),
    (64, 3, 1500, 4, 63, 0.3),
    (3, 5, 300_000, 8, 20_001, 0.05),       # 128 taus and more
    (4, 4, 1_200_000, 4, 100_003, 0.02),    # 18 levels
])
def test_sums_equal_numpy(xmt, W, H, F, dpl, piece, filled):
    import torch
    rng = np.random.default_rng(F + dpl)
    P = W * H
    # payloads (u32 indices, u16 values): number 0 is empty, the others hold
    # up to half of the pixels
    pool = np.zeros((41, P), np.int64)
    raw, off, dl = b"", [], []
    for k in range(41):
        idx = rng.permutation(P)[:0 if k == 0 else 1 + P // 2].astype(np.uint32)
        pool[k, idx] = rng.integers(1, 300, len(idx))
        off.append(len(raw))
        dl.append(len(idx))
        raw += idx.tobytes() + pool[k, idx].astype(np.uint16).tobytes()
    pick = np.where(rng.random(F) < filled, rng.integers(1, 41, F), 0)
    buf = torch.frombuffer(bytearray(raw), dtype=torch.uint8).cuda()
    torch.cuda.synchronize()
    off, dl = np.array(off, np.int64)[pick], np.array(dl, np.uint32)[pick]
    ones = np.ones((H, W), np.int32)
    print("stream", W, H, F, dpl, flush=True)
    s = xmt.Stream(W, H, F, dpl, ones, ones)
    for a in range(0, F, piece):
        b = min(F, a + piece)
        s.push_imm_device(buf.data_ptr(), buf.numel(), off[a:b], dl[a:b])
    s.snapshot()
    got = s.sums()
    levels, taus = xmt.delays_per_level(F, dpl)
    s.close()
    want = level_sums(pool[pick], taus, levels)
    for g, w in zip(got, want):
        assert g.shape == w.shape and np.array_equal(g, w)
