"""Dark image on the device: mean and deviation bit-equal to the oracle's
Welford pass in frame order, from a host and a device ingest, up to more frames
than one launch takes and with values above 32767."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,darks", [(16, 16, 1), (31, 9, 3), (20, 13, 64), (20, 13, 65), (9, 7, 130)])
def test_dark_image_bits(xmt, orc, W, H, darks):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(darks)
    F = 40
    dq, sq = synth.annular_qmaps(W, H, 4, 2)
    dark = rng.integers(0, 65536, (darks, W * H)).astype(np.uint16)
    raw = np.concatenate([dark, rng.integers(0, 65536, (F, W * H)).astype(np.uint16)])
    imm = synth.imm_bytes_dense(raw, W, H)
    avg = np.zeros(W * H)
    dev = np.zeros(W * H)
    for i in range(darks):
        x = dark[i].astype(np.float64)
        prev = avg.copy()
        avg = avg + (x - avg) / (i + 1)
        dev = dev + (x - prev) * (x - avg)
    dev = np.sqrt(dev / darks)
    r = orc.run_exact(imm, dq, sq, F, 4, darks=darks, lld=2.5, sigma=1.25)
    for device in (False, True):
        print(f"dark image {W}x{H} darks={darks} device={device}", flush=True)
        plan = xmt.Plan(W, H, F, 4, dq, sq, dark_frames=darks, lld=2.5, sigma=1.25)
        if device:
            buf = torch.from_numpy(np.frombuffer(imm, np.uint8).copy()).cuda()
            torch.cuda.synchronize()
            idx = xmt.imm_index(imm)
            plan.ingest_imm_device(buf.data_ptr(), buf.numel(), idx["payload_off"], idx["dlen"], compressed=False)
        else:
            plan.ingest_imm(imm)
        plan.execute()
        g, a, b = plan.sums()
        got = np.zeros((2, W * H))
        xmt.check(xmt.lib().xpcs_mt_read_dark(plan._h, xmt._p(got[0]), xmt._p(got[1])))
        plan.close()
        assert np.array_equal(got[0], avg) and np.array_equal(got[1], dev)
        assert np.array_equal(a, r["IP"]) and np.array_equal(b, r["IF"]) and np.array_equal(g, r["G2"])
