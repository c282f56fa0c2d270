"""Workloads of the multi-tau correlator, from the smallest job to the largest.

Every case is what a beamline program does with one measurement: it holds a plan
for its detector and q-partition, receives the frames (an IMM image in GPU memory
or, for files, in host memory), and asks for the correlation.  The q-maps are
nested annuli; the counts are Poisson draws of a speckle intensity (a complex
Ornstein-Uhlenbeck field per speckle, speckles of 2 x 2 pixels, correlation times
log-spaced over the detector radius), so that rows, repeats and empty pixels come
in the proportions of photon-counting (sparse) or integrating (dense) detectors.

kinds
  sparse    compressed IMM image in GPU memory -> g2, stderr (options: averaged
            frames, flat field, side statistics, normalize_by_framesum)
  host      compressed IMM file bytes in host memory -> g2, stderr
  dense     uncompressed IMM image in GPU memory -> g2, stderr (options: dark
            frames with threshold, flat field)
  stream    frames pushed a few at a time, g2 read at regular snapshots
  batch     many uneven sparse jobs, launched together, g2 of each
  tt        two-time matrices and their diagonals (sparse or dense frames)
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("xpcs-eigen_amd"))
import xpcs_mt  # noqa: E402

HEADER = 1024


def listed():
    return [
        # one short exposure of a small region of interest: latency of a call
        dict(name="sparse-roi128", kind="sparse", w=128, h=128, frames=500, dpl=4, mu=0.02, S=9, Q=3),
        # the command line tool's path: a small file's bytes in host memory
        dict(name="file-256", kind="host", w=256, h=256, frames=1000, dpl=4, mu=0.012, S=18, Q=6),
        # the headline job: megapixel photon-counting detector, 10,000 frames
        dict(name="sparse-1mpx", kind="sparse", w=1024, h=1024, frames=10000, dpl=8, mu=0.005, S=36, Q=12),
        # an odd-sized detector with everything on: flat field, frames averaged
        # in pairs, frame sums and partition means recorded
        dict(name="sparse-ragged", kind="sparse", w=517, h=389, frames=3501, dpl=8, mu=0.008, S=30, Q=10,
             avg=2, flat=True, side=True),
        # a bright sample on a counting detector: rows of hundreds of events
        dict(name="sparse-bright", kind="sparse", w=600, h=600, frames=12000, dpl=4, mu=0.025, S=27, Q=9),
        # incident-flux correction: every frame scaled by its sum
        dict(name="framesum-640", kind="sparse", w=640, h=480, frames=5000, dpl=8, mu=0.01, S=24, Q=8,
             fsnorm=True),
        # integrating detector, two dark frames, 20,000 frames
        dict(name="dense-512", kind="dense", w=512, h=512, frames=20000, dpl=4, mu=5.0, S=27, Q=9, darks=2),
        # integrating detector cropped to an odd region, flat field, no darks
        dict(name="dense-ragged", kind="dense", w=333, h=251, frames=3001, dpl=8, mu=3.0, S=18, Q=6, flat=True),
        # a live view: frames arrive 16 at a time, g2 shown every 64 frames
        dict(name="live-256", kind="stream", w=256, h=256, frames=1024, dpl=4, mu=0.01, S=18, Q=6,
             push=16, every=64),
        # a night's queue of uneven jobs in one launch
        dict(name="batch-16", kind="batch", jobs=16, wmin=128, wmax=512, fmin=500, fmax=6000, seed0=4000),
        # two-time maps of two q-bins, photon counting
        dict(name="twotime-sparse", kind="tt", w=512, h=512, frames=2048, dpl=8, mu=0.02, S=18, Q=6,
             dense=False, nq=2, window=64, smoothing=1),
        # two-time maps of two q-bins, integrating detector
        dict(name="twotime-dense", kind="tt", w=256, h=256, frames=2048, dpl=4, mu=5.0, S=18, Q=6, darks=2,
             dense=True, nq=2, window=64, smoothing=1),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sparse", "sparse", "sparse", "host", "dense", "dense", "stream", "batch", "tt"])
    dpl = rng.choice([4, 8])
    Q = rng.randint(2, 12)
    ring = dict(dpl=dpl, S=3 * Q, Q=Q)
    if kind in ("sparse", "host"):
        while True:
            w = _logint(rng, 128, 1024)
            h = max(96, int(w * rng.uniform(0.6, 1.0)))
            frames = _logint(rng, 500, 12000)
            mu = math.exp(rng.uniform(math.log(0.002), math.log(0.03)))
            avg = rng.choice([1, 1, 1, 2])
            ev = w * h * frames * mu * avg
            if ev > (2e7 if kind == "host" else 6e7) or mu * avg * frames < 8:
                continue
            c = dict(kind=kind, w=w, h=h, frames=frames, mu=mu, **ring)
            if kind == "sparse":
                c["avg"] = avg
                c["flat"] = rng.random() < 0.25
                c["side"] = rng.random() < 0.25
                c["fsnorm"] = rng.random() < 0.2
            elif avg != 1:
                continue
            return c
    if kind == "dense":
        while True:
            w = _logint(rng, 128, 512)
            h = max(96, int(w * rng.uniform(0.6, 1.0)))
            frames = _logint(rng, 500, 12000)
            if w * h * frames > 1.5e9:
                continue
            darks = rng.choice([0, 2, 3])
            return dict(kind="dense", w=w, h=h, frames=frames, mu=math.exp(rng.uniform(math.log(1.0), math.log(60.0))),
                        darks=darks, flat=darks == 0 and rng.random() < 0.4, **ring)
    if kind == "stream":
        w = _logint(rng, 128, 512)
        push = rng.randint(4, 40)
        return dict(kind="stream", w=w, h=max(96, int(w * rng.uniform(0.6, 1.0))), frames=rng.randint(256, 1500),
                    mu=math.exp(rng.uniform(math.log(0.004), math.log(0.03))), push=push,
                    every=push * rng.randint(2, 6), **ring)
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(4, 16), wmin=128, wmax=rng.randint(256, 512), fmin=500,
                    fmax=rng.randint(2000, 6000), seed0=rng.randint(1, 100000))
    dense = rng.random() < 0.5
    w = _logint(rng, 128, 256 if dense else 512)
    return dict(kind="tt", w=w, h=max(96, int(w * rng.uniform(0.6, 1.0))), frames=rng.randint(500, 2048), dense=dense,
                mu=rng.uniform(1.0, 20.0) if dense else rng.uniform(0.01, 0.03), darks=2 if dense else 0,
                nq=rng.randint(1, 2), window=rng.choice([16, 64]), smoothing=rng.choice([0, 1, 1, 2]), **ring)


# ---- inputs ---------------------------------------------------------------------

def _qmaps(w, h, S, Q):
    """(dqmap, sqmap) int32 [h, w]: nested annuli of radius w / 2, 0 outside."""
    y, x = np.mgrid[0:h, 0:w].astype(np.float64)
    r = np.sqrt((x - (w - 1) / 2.0) ** 2 + (y - (h - 1) / 2.0) ** 2) / (w / 2.0)
    s = np.where(r < 1.0, 1 + np.floor(S * r), 0).astype(np.int32)
    q = np.where(s > 0, 1 + (s - 1) // (S // Q), 0).astype(np.int32)
    return q, s


def _counts(w, h, frames, mu, seed, tau=(2.0, 2000.0), step=256):
    """Blocks (first frame, int32 counts [n, h * w]) on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    gw, gh = (w + 1) // 2, (h + 1) // 2
    yy = torch.arange(gh, device="cuda", dtype=torch.float32)[:, None] / gh - 0.5
    xx = torch.arange(gw, device="cuda", dtype=torch.float32)[None, :] / gw - 0.5
    rad = (2.0 * torch.sqrt(yy * yy + xx * xx)).clamp(max=1.0).reshape(-1)
    a = torch.exp(-1.0 / (tau[0] * (tau[1] / tau[0]) ** (1.0 - rad)))
    b = torch.sqrt((1.0 - a * a) * 0.5)
    e = torch.randn((2, gh * gw), generator=g, device="cuda") * math.sqrt(0.5)
    t = 0
    while t < frames:
        n = min(step, frames - t)
        xi = torch.randn((n, 2, gh * gw), generator=g, device="cuda").mul_(b)
        E = torch.empty_like(xi)
        for k in range(n):
            torch.addcmul(xi[k], a, e, out=E[k])
            e = E[k]
        e = e.clone()
        lam = (E * E).sum(1).mul_(mu).view(n, gh, 1, gw, 1).expand(n, gh, 2, gw, 2).reshape(n, 2 * gh, 2 * gw)
        c = torch.poisson(lam[:, :h, :w].contiguous(), generator=g).clamp_(max=60000.0)
        yield t, c.view(n, h * w).to(torch.int32)
        t += n


def _headers(compression, w, h, dlen, first):
    n = len(dlen)
    hd = np.zeros((n, HEADER), np.uint8)

    def put(off, v, dt):
        a = np.empty((n, 1), dt)
        a[:, 0] = v
        hd[:, off:off + a.itemsize] = a.view(np.uint8)
    t = np.arange(first, first + n)
    put(4, compression, np.int32)
    put(108, h, np.int32)
    put(112, w, np.int32)
    put(116, 2, np.int32)
    put(128, t * 1.0e-3, np.float64)
    put(152, dlen, np.uint32)
    put(160, t, np.int32)
    put(616, 12, np.int32)
    put(620, t, np.int32)
    return torch.from_numpy(hd.view(np.int16)).cuda()


def _imm_sparse(w, h, blocks):
    """Compressed IMM image on the GPU: (uint8 tensor, payload offsets, event counts)."""
    parts, offs, dls = [], [], []
    pos = 0
    for t0, c in blocks:
        n = c.shape[0]
        flat = torch.nonzero(c.view(-1)).view(-1)
        val = c.view(-1)[flat].to(torch.int16)
        fr = flat // (w * h)
        px = (flat - fr * (w * h)).to(torch.int32)
        dl = torch.bincount(fr, minlength=n)
        rec = HEADER // 2 + 3 * dl                    # in 16-bit units
        start = torch.cumsum(rec, 0) - rec
        first = torch.cumsum(dl, 0) - dl
        buf = torch.empty(int(rec.sum()), dtype=torch.int16, device="cuda")
        dlh = dl.cpu().numpy()
        sth = start.cpu().numpy()
        buf[(start[:, None] + torch.arange(HEADER // 2, device="cuda")).view(-1)] = \
            _headers(6, w, h, dlh, t0).view(-1)
        rank = torch.arange(flat.numel(), device="cuda") - first[fr]
        body = start[fr] + HEADER // 2
        pv = px.view(torch.int16).view(-1, 2)
        buf[body + 2 * rank] = pv[:, 0]
        buf[body + 2 * rank + 1] = pv[:, 1]
        buf[body + 2 * dl[fr] + rank] = val
        parts.append(buf)
        offs.append(2 * (pos + sth) + HEADER)
        dls.append(dlh)
        pos += int(rec.sum())
    imm = torch.cat(parts).view(torch.uint8)
    return imm, np.concatenate(offs).astype(np.int64), np.concatenate(dls).astype(np.uint32)


def _dark(npix, n, seed):
    """n dark frames int32 [n, npix]: readout noise about a per-pixel offset."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2 + 1)
    base = (2.0 + 0.5 * torch.randn(npix, generator=g, device="cuda"))
    d = base[None, :] + 0.3 * torch.randn((n, npix), generator=g, device="cuda")
    return d.round().clamp_(min=0).to(torch.int32)


def _imm_dense(w, h, frames, blocks, darks, seed):
    npix = w * h
    unit = HEADER // 2 + npix
    buf = torch.empty((frames + darks, unit), dtype=torch.int16, device="cuda")
    off = 0
    if darks:
        d = _dark(npix, darks, seed)
        buf[:darks, :HEADER // 2] = _headers(0, w, h, np.full(darks, npix), 0)
        buf[:darks, HEADER // 2:] = d.to(torch.int16)
        off = d[0]
    for t0, c in blocks:
        n = c.shape[0]
        buf[darks + t0:darks + t0 + n, :HEADER // 2] = _headers(0, w, h, np.full(n, npix), darks + t0)
        buf[darks + t0:darks + t0 + n, HEADER // 2:] = (c + off).clamp_(max=65535).to(torch.int16)
    offs = np.arange(frames + darks, dtype=np.int64) * unit * 2 + HEADER
    return buf.view(-1).view(torch.uint8), offs, np.full(frames + darks, npix, np.uint32)


def _flat(c, seed):
    if not c.get("flat"):
        return None
    return np.random.default_rng(seed).uniform(0.8, 1.25, (c["h"], c["w"]))


THRESHOLD = dict(lld=1.0, sigma=2.0)


def _plan(c, seed):
    q, s = _qmaps(c["w"], c["h"], c["S"], c["Q"])
    kw = {}
    if c.get("darks"):
        kw = dict(dark_frames=c["darks"], **THRESHOLD)
    return xpcs_mt.Plan(c["w"], c["h"], c["frames"], c["dpl"], q, s, average=c.get("avg", 1), flatfield=_flat(c, seed),
                        side_stats=c.get("side", False), normalize_by_framesum=c.get("fsnorm", False), **kw)


def _is_dense(c):
    return c["kind"] == "dense" or c.get("dense", False)


def _image(c, seed):
    w, h = c["w"], c["h"]
    if _is_dense(c):
        return _imm_dense(w, h, c["frames"], _counts(w, h, c["frames"], c["mu"], seed), c.get("darks", 0), seed)
    return _imm_sparse(w, h, _counts(w, h, c["frames"] * c.get("avg", 1), c["mu"], seed))


def _batch_jobs(c):
    jobs = []
    for j in range(c["jobs"]):
        r = random.Random(c["seed0"] + j)
        Q = r.randint(2, 12)
        jobs.append(dict(kind="sparse", w=r.randint(c["wmin"], c["wmax"]), frames=r.randint(c["fmin"], c["fmax"]),
                         mu=math.exp(r.uniform(math.log(0.002), math.log(0.05))), dpl=r.choice([4, 8]), S=3 * Q, Q=Q))
        jobs[-1]["h"] = jobs[-1]["w"]
    return jobs


def _qbins(c):
    return list(range(2, 2 + c["nq"]))


def prepare(case, seed):
    c = case
    if c["kind"] == "batch":
        plans, keep = [], []
        batch = xpcs_mt.Batch()
        for j, job in enumerate(_batch_jobs(c)):
            imm, off, dl = _image(job, seed * 100 + j)
            torch.cuda.synchronize()
            plan = _plan(job, seed)
            plan.ingest_imm_device(imm.data_ptr(), imm.numel(), off, dl, compressed=True)
            batch.add(plan)
            plans.append(plan)
            keep.append(imm)
        return dict(case=c, batch=batch, plans=plans, keep=keep)
    imm, off, dl = _image(c, seed)
    torch.cuda.synchronize()
    if c["kind"] == "host":
        return dict(case=c, plan=_plan(c, seed), file=imm.cpu().numpy())
    if c["kind"] == "stream":
        q, s = _qmaps(c["w"], c["h"], c["S"], c["Q"])
        return dict(case=c, imm=imm, off=off, dl=dl, q=q, s=s)
    return dict(case=c, plan=_plan(c, seed), imm=imm, off=off, dl=dl)


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "batch":
        state["batch"].execute()
        return [p.g2() for p in state["plans"]]
    if kind == "host":
        plan = state["plan"]
        plan.ingest_imm(state["file"])
        plan.execute()
        return plan.g2()
    imm, off, dl = state["imm"], state["off"], state["dl"]
    if kind == "stream":
        out = []
        live = xpcs_mt.Stream(c["w"], c["h"], c["frames"], c["dpl"], state["q"], state["s"])
        shown = 0
        for f in range(0, c["frames"], c["push"]):
            e = min(f + c["push"], c["frames"])
            live.push_imm_device(imm.data_ptr(), imm.numel(), off[f:e], dl[f:e])
            if e - shown >= c["every"] or e == c["frames"]:
                live.snapshot()
                out.append(live.g2())
                shown = e
        live.close()
        return out
    plan = state["plan"]
    plan.ingest_imm_device(imm.data_ptr(), imm.numel(), off, dl, compressed=not _is_dense(c))
    if kind == "tt":
        r = plan.twotime(_qbins(c), smoothing=c["smoothing"], window=c["window"])
        return r["c2t"] + [r["g2full"], r["g2partials"]] + ([r["sg"]] if r["sg"] is not None else [])
    plan.execute()
    out = list(plan.g2())
    if c.get("side"):
        s = plan.side(frame_sum=True)
        out += [s["pixel_sum"], s["partition_mean"], s["frame_sum"]]
    return out


# ---- work and exact results -------------------------------------------------------

def _schedule(frames, dpl):
    """[(level, lag in level frames)]: 2 dpl lags at level 0, dpl at each further
    level of step 2^level, as long as the next two steps fit the frames."""
    if frames < 2 * dpl:
        top = 0
    else:
        top = int(math.floor(math.log2(frames) - math.log2(1.0 + 1.0 / dpl)) - math.log2(dpl))
    out, tau = [], 0
    for L in range(top + 1):
        for _ in range(2 * dpl if L == 0 else dpl):
            if tau + (2 << L) > frames:
                break
            tau += 1 << L
            out.append((L, tau >> L))
    return out


def _one_work(c):
    q, _ = _qmaps(c["w"], c["h"], c["S"], c["Q"])
    F, npix, P = c["frames"], c["w"] * c["h"], int((q > 0).sum())
    if _is_dense(c):
        nbytes = 2.0 * npix * (F + c.get("darks", 0))
    else:
        nbytes = 6.0 * npix * F * c.get("avg", 1) * c["mu"] / (1.0 + c["mu"])
    if c["kind"] == "tt":
        Pq = float(np.isin(q, _qbins(c)).sum())
        nbytes += 8.0 * c["nq"] * F * F
        occ = 1.0 if _is_dense(c) else c["mu"] / (1.0 + c["mu"])
        return nbytes, Pq * F * (F + 1.0) * occ * occ
    flops = 0.0
    taus = _schedule(F, c["dpl"])
    for L, lag in taus:
        m = c["mu"] * c.get("avg", 1) * 2.0 ** L
        occ = 1.0 if _is_dense(c) else m / (1.0 + m)
        flops += 2.0 * P * max((F >> L) - lag, 0) * occ * occ
    nbytes += 16.0 * len(taus) * c["Q"]
    if c.get("side"):
        nbytes += 4.0 * npix + 8.0 * F
    return nbytes, flops


def work(case):
    jobs = _batch_jobs(case) if case["kind"] == "batch" else [case]
    b, f = zip(*(_one_work(j) for j in jobs))
    return {"bytes": sum(b), "flops": sum(f)}


def _values(c, seed):
    """Values of the mapped pixels [F, P] (counts, frames averaged in sums;
    dense frames times the number of darks, after subtraction and threshold)
    and, per pixel, static bin, dynamic bin, and raster index; value scale."""
    w, h, F, avg = c["w"], c["h"], c["frames"], c.get("avg", 1)
    q, s = _qmaps(w, h, c["S"], c["Q"])
    pix = np.flatnonzero(q.reshape(-1) > 0)
    idx = torch.as_tensor(pix, device="cuda")
    darks = c.get("darks", 0)
    X = torch.empty((F * avg, pix.size), dtype=torch.int32 if darks else torch.int16, device="cuda")
    if darks:
        d = _dark(w * h, darks, seed)[:, idx].double()
        t = THRESHOLD["lld"] + THRESHOLD["sigma"] * d.std(0, unbiased=False)
        thr = torch.floor(darks * t.float().double()).clamp(min=0)
        dsum = d.sum(0)
        d0 = _dark(w * h, darks, seed)[0, idx]
    for t0, b in _counts(w, h, F * avg, c["mu"], seed):
        v = b[:, idx]
        if darks:
            y = darks * (v + d0).clamp_(max=65535).double() - dsum
            v = torch.where(y > thr, y, torch.zeros_like(y))
        X[t0:t0 + v.shape[0]] = v.to(X.dtype)
    return X, s.reshape(-1)[pix], q.reshape(-1)[pix], pix, 1.0 / (avg * max(darks, 1))


def _exact_g2(c, X, sb, qb, flat, frames):
    """g2 and stderr [T, Q] in 64 bits."""
    taus = _schedule(frames, c["dpl"])
    S, Q, T, avg = c["S"], c["Q"], len(taus), c.get("avg", 1)
    P = X.shape[1]
    dev = X.device
    wt = torch.ones(P, dtype=torch.float64, device=dev) if flat is None else torch.as_tensor(flat, device=dev)
    fw = None
    if c.get("fsnorm"):
        fs = torch.zeros(frames, dtype=torch.float64, device=dev)
        for p0 in range(0, P, 16384):
            x = X[:, p0:p0 + 16384].double()
            if avg > 1:
                x = x.view(frames, avg, -1).sum(1)
            fs += (x * wt[p0:p0 + 16384]).sum(1)
        fw = torch.where(fs > 0, fs.mean() / fs, torch.zeros_like(fs))
    sums = torch.zeros((3, S, T), dtype=torch.float64, device=dev)
    sidx = torch.as_tensor(sb.astype(np.int64) - 1, device=dev)
    qidx = torch.as_tensor(qb.astype(np.int64) - 1, device=dev)
    npx = torch.bincount(qidx, minlength=Q).double()
    nsx = torch.bincount(sidx, minlength=S).double()
    ratios = torch.zeros((T, P), dtype=torch.float64, device=dev)
    step = max(256, int(2.5e8 // frames))
    for p0 in range(0, P, step):
        x = X[:frames * avg, p0:p0 + step].double()
        if avg > 1:
            x = x.view(frames, avg, -1).sum(1)
        if fw is not None:
            x = x * fw[:, None]
        w = wt[p0:p0 + step]
        si = sidx[p0:p0 + step]
        level = 0
        for i, (L, lag) in enumerate(taus):
            while level < L:
                n = x.shape[0] // 2
                x = x[0:2 * n:2] + x[1:2 * n:2]
                level += 1
            N = x.shape[0] - lag
            a, b = x[:N], x[lag:]
            g, ip, jf = (a * b).sum(0), a.sum(0), b.sum(0)
            r = N * g / (ip * jf)
            ratios[i, p0:p0 + step] = torch.where((w == 0) | torch.isnan(r), torch.zeros_like(r), r)
            sums[0, :, i].index_add_(0, si, g * w * w)
            sums[1, :, i].index_add_(0, si, ip * w)
            sums[2, :, i].index_add_(0, si, jf * w)
    N = torch.tensor([(frames >> L) - lag for L, lag in taus], dtype=torch.float64, device=dev)
    g2s = nsx[:, None] * N * sums[0] / (sums[1] * sums[2])
    ok = ~torch.isnan(g2s)
    v = torch.where(ok, g2s, torch.zeros_like(g2s)).view(Q, S // Q, T).sum(1)
    g2 = v / ok.view(Q, S // Q, T).sum(1)
    se = torch.zeros((T, Q), dtype=torch.float64, device=dev)
    for q in range(Q):
        se[:, q] = ratios[:, qidx == q].var(1, unbiased=False).sqrt() / npx[q].sqrt()
    return g2.T.contiguous().cpu().numpy(), se.cpu().numpy()


def _exact_tt(c, X, sb, qb, scale):
    F, wsz = c["frames"], c["window"]
    total = (F - wsz) // wsz
    c2t, sgs = [], []
    nq = c["nq"]
    full = np.zeros((F, nq))
    part = np.zeros((wsz, total, nq))
    for i, q in enumerate(_qbins(c)):
        sel = np.flatnonzero(qb == q)
        x = X[:, torch.as_tensor(sel, device=X.device)].double() * scale      # [F, Pq]
        if c["smoothing"]:
            bins = sb[sel] if c["smoothing"] == 1 else np.zeros(sel.size, np.int32)
            for b in np.unique(bins):
                k = torch.as_tensor(np.flatnonzero(bins == b), device=X.device)
                m = x[:, k].mean(1)
                sgs.append(m.cpu().numpy())
                x[:, k] = x[:, k] / torch.where(m != 0, m, torch.ones_like(m))[:, None]
        G = torch.triu(x @ x.T) / sel.size
        cols = torch.arange(F, device=X.device)
        lag = cols[None, :] - cols[:, None]
        s = torch.zeros(F, dtype=torch.float64, device=X.device)
        up = lag >= 0
        s.index_add_(0, lag[up], G[up])
        full[:, i] = (s / (F - cols)).cpu().numpy()
        for f in range(wsz):
            d = torch.nn.functional.pad(torch.diagonal(G, f), (0, f))[:total * wsz]
            part[f, :, i] = (d.view(total, wsz).sum(1) / wsz).cpu().numpy()
        c2t.append(G.cpu().numpy())
    return c2t + [full, part] + ([np.stack(sgs)] if sgs else [])


def exact(case, seed):
    c = case
    if c["kind"] == "batch":
        out = []
        for j, job in enumerate(_batch_jobs(c)):
            X, sb, qb, _, _ = _values(job, seed * 100 + j)
            out.append(_exact_g2(job, X, sb, qb, None, job["frames"]))
        return out
    X, sb, qb, pix, scale = _values(c, seed)
    flat = _flat(c, seed)
    fp = None if flat is None else flat.reshape(-1)[pix]
    if c["kind"] == "tt":
        return _exact_tt(c, X, sb, qb, scale)
    if c["kind"] == "stream":
        out, shown = [], 0
        for f in range(0, c["frames"], c["push"]):
            e = min(f + c["push"], c["frames"])
            if e - shown >= c["every"] or e == c["frames"]:
                out.append(_exact_g2(c, X[:e], sb, qb, None, e))
                shown = e
        return out
    out = list(_exact_g2(c, X, sb, qb, fp, c["frames"]))
    if c.get("side"):
        F, npix = c["frames"], c["w"] * c["h"]
        wt = torch.ones(pix.size, dtype=torch.float64, device=X.device) if fp is None else \
            torch.as_tensor(fp, device=X.device)
        tot = torch.zeros(pix.size, dtype=torch.float64, device=X.device)
        fs = torch.zeros(F * c.get("avg", 1), dtype=torch.float64, device=X.device)
        for f in range(0, X.shape[0], 256):
            b = X[f:f + 256].double()
            tot += b.sum(0)
            fs[f:f + 256] = (b * wt).sum(1)
        val = (tot * wt * scale / F).cpu().numpy()
        ps = np.zeros(npix)
        ps[pix] = val
        pm = np.bincount(sb - 1, weights=val, minlength=c["S"]) / np.bincount(sb - 1, minlength=c["S"])
        fsum = fs.view(F, -1).sum(1).cpu().numpy() * scale / npix
        out += [ps, pm, np.stack([np.arange(1.0, F + 1.0), fsum])]
    if c["kind"] == "host":
        out = tuple(out)
    return out
