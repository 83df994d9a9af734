"""The work that users of fdt_amd have it do, as timed cases.

listed() is the fixed set, draw(rng) gives further cases of the same ranges.
A case is a dict of plain values; its "kind" names the path:

  call     run_xfibres on a handful of voxels: a context made, the whole
           pipeline run and everything read back in one call
  run      one part of a volume through a kept context, from page-locked host
           buffers: upload, LM initialisation, chains, finishing, download
           (what xfibres_gpu and bedpostx_gpu do); with rician, f0 and
           --gradnonlin as options
  fit      the LM initialisation alone, parameters read back
  chains   the chains and the finishing from start values in hand (a caller
           with its own initialisation)
  spatial  the CPU xfibres neighbour initialisation: wavefronts of short
           launches over a grid
  queue    four volumes of different acquisition, model and fibre count run
           together (single-subject batches)
  learned  the learned start with the short burn-in and the plain fallback
  infer    the network alone: start values of resident voxels
  train    steps of the network's training from given weights, the trained
           ones read back

Signals are drawn from the ball-and-sticks family with Rician noise, as in
fdt_amd.synth, but on the GPU.  Jump counts are the defaults of xfibres
(burn-in 1000, 1250 recorded jumps, every 25th kept) unless a case says
otherwise.
"""
import math
import os

import numpy as np
import torch

import fdt_amd
from fdt_amd import synth

DEV = "cuda"
R_TRUE = 0.13  # zeppelin ratio of the model-3 signals (the mean of the R prior)
# the queue's four volumes: volumes, shells, model, fibres
QUEUE_MIX = ((33, 1, 1, 1), (69, 1, 2, 2), (145, 3, 2, 3), (288, 3, 3, 3))
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(fdt_amd.__file__)), "weights", "surrogate_c1_model2_nf3.npz")


def listed():
    return [
        # the smallest use: a region of interest of 48 voxels of a single-shell scan, one call (latency, allocations)
        dict(name="call_roi_48", kind="call", N=69, shells=1, model=1, nf=2, nvox=48),
        # a single-shell slice of 2,000 voxels, two fibres, the ball-and-sticks model
        dict(name="run_single_shell_2k", kind="run", N=69, shells=1, model=1, nf=2, nvox=2000),
        # a whole multi-shell brain at 2 mm: 250,968 voxels, 288 volumes, model 2, three fibres (the headline workload)
        dict(name="run_multi_shell_brain", kind="run", N=288, shells=3, model=2, nf=3, nvox=250968),
        # one of 32 parts of a 145-volume scan with gradient nonlinearity correction; a ragged voxel count
        dict(name="run_gradnonlin_part", kind="run", N=145, shells=3, model=2, nf=3, nvox=7843, grad=True),
        # a long acquisition (432 volumes) with a noise-floor compartment (--f0: FP64 fits and the refit)
        dict(name="run_f0_long", kind="run", N=432, shells=3, model=2, nf=2, nvox=3001, f0=True),
        # the initialisation alone on a few slices of the multi-shell volume
        dict(name="fit_multi_shell_20k", kind="fit", N=288, shells=3, model=2, nf=3, nvox=20011),
        # zeppelins with the Rician noise model (high-resolution data), chains alone
        dict(name="chains_rician_16k", kind="chains", N=288, shells=3, model=3, nf=3, nvox=16384, rician=True),
        # the neighbour initialisation on a small single-shell slab
        dict(name="spatial_slab", kind="spatial", N=69, shells=1, model=1, nf=2, nx=18, ny=16, nz=5),
        # four different small volumes in one batch
        dict(name="queue_mixed_4x6k", kind="queue", nvox=6000),
        # the learned start on a few slices of the multi-shell volume (burn-in 200, as the workload specifies it)
        dict(name="learned_30k", kind="learned", nvox=30000),
        # start values from the network for the whole multi-shell brain
        dict(name="infer_brain", kind="infer", N=288, nvox=250968),
        # eight training steps of the network at the batch size of its training driver
        dict(name="train_8x1024", kind="train", N=288, batch=1024, steps=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _options(rng, c):
    """acquisition, model and fibre count of a drawn case"""
    c["N"] = rng.choice([33, 69, 145, 288, rng.randrange(20, 289), rng.randrange(289, 440)])
    c["shells"] = 1 if c["N"] < 70 else 3
    c["model"] = rng.choice([1, 2, 2, 3]) if c["shells"] == 3 else rng.choice([1, 1, 2])
    c["nf"] = rng.choice([1, 2, 3, 3]) if c["N"] > 40 else rng.choice([1, 2])
    if rng.random() < 0.25:
        c["rician"] = True
    return c


def _us_per_voxel(c):
    """a rough cost, to keep drawn cases below the largest listed one"""
    us = 6.0 * c["N"] / 288 * (c["nf"] + 1) / 4 * (1.6 if c["model"] == 3 else 1.0) * (2.2 if c.get("rician") else 1.0)
    return us * (2.0 if c["N"] > 288 else 1.0) + (4.0 if c.get("f0") else 1.5)


def draw(rng):
    kind = rng.choice(["call", "run", "run", "run", "fit", "chains", "chains", "spatial", "queue", "learned", "infer", "train"])
    c = dict(kind=kind)
    if kind == "call":
        c.update(N=rng.choice([33, 69, 145, rng.randrange(20, 150)]), shells=1, model=rng.choice([1, 2]),
                 nf=rng.choice([1, 2]), nvox=_log_int(rng, 16, 900))
    elif kind in ("run", "fit", "chains"):
        _options(rng, c)
        if kind != "chains" and not c.get("rician") and rng.random() < 0.25:
            c[rng.choice(["f0", "grad"])] = True
        c["nvox"] = _log_int(rng, 500, min(60000, int(300e3 / _us_per_voxel(c))))
    elif kind == "spatial":
        c.update(N=rng.choice([33, 69, rng.randrange(20, 100)]), shells=1, model=1, nf=rng.choice([1, 2]),
                 nx=rng.randrange(8, 22), ny=rng.randrange(8, 18), nz=rng.randrange(2, 7))
    elif kind == "queue":
        c["nvox"] = _log_int(rng, 500, 12000)
    elif kind == "learned":
        c["nvox"] = _log_int(rng, 1000, 60000)
    elif kind == "infer":
        c.update(N=rng.choice([69, 145, 288, rng.randrange(33, 433)]), nvox=_log_int(rng, 1000, 250000))
    else:
        c.update(N=rng.choice([69, 145, 288, rng.randrange(33, 433)]), batch=rng.choice([256, 1000, 1024, 2048, 4096]),
                 steps=rng.randrange(2, 9))
    return c


# ------------------------------------------------------------------ inputs

def _acquisition(N, shells, seed):
    """bvals [N] and bvecs [3][N]: one b = 0 volume in 16, the rest on one shell (b = 1000) or three"""
    n0 = max(2, (N + 8) // 16)
    dirs = [(N - n0) // shells + (1 if i < (N - n0) % shells else 0) for i in range(shells)]
    g = np.random.Generator(np.random.Philox(key=[seed, 17]))
    return synth.acquisition(n0, [(1000.0 * (i + 1), n) for i, n in enumerate(dirs)], g)


def _gen(seed, stream=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 64 + stream)


def _unit(g, *shape):
    v = torch.randn(*shape, 3, device=DEV, generator=g)
    return v / v.norm(dim=-1, keepdim=True)


def _host(t):
    """a page-locked numpy copy of a device tensor"""
    t = t.contiguous()
    a = fdt_amd.pinned_empty(tuple(t.shape))
    torch.from_numpy(a).copy_(t)
    return a


def _signals(bvals, bvecs, model, nvox, g, grad=None):
    """noisy signals [nvox][N] float32 on the GPU and the truth they come from: one to three sticks (one or two on
    one shell) at 30 to 90 degrees, SNR 25 (20 on one shell)"""
    b = torch.tensor(bvals, dtype=torch.float32, device=DEV)
    gv = torch.tensor(bvecs, dtype=torch.float32, device=DEV)
    single = len(set(bvals.tolist())) <= 2
    u = lambda lo, hi, *s: lo + (hi - lo) * torch.rand(*s, device=DEV, generator=g)
    S0 = u(800.0, 1200.0, nvox)
    d = u(0.8e-3, 2.0e-3, nvox)
    dstd = torch.minimum(d * u(0.1, 0.5, nvox), torch.full_like(d, 0.0039))
    nfib = torch.randint(1, 3 if single else 4, (nvox,), device=DEV, generator=g)
    w = -torch.log(u(1e-6, 1.0, nvox, 3)) * (torch.arange(3, device=DEV)[None] < nfib[:, None])
    f = w / w.sum(1, keepdim=True) * u(0.3, 0.8, nvox)[:, None]
    f = f.sort(dim=1, descending=True).values
    x = _unit(g, nvox, 3)
    for k in (1, 2):
        ang = u(math.pi / 6, math.pi / 2, nvox)[:, None]
        p = x[:, k] - (x[:, k] * x[:, 0]).sum(1, keepdim=True) * x[:, 0]
        x[:, k] = torch.cos(ang) * x[:, 0] + torch.sin(ang) * p / p.norm(dim=1, keepdim=True)
    y = torch.empty(nvox, b.numel(), device=DEV)
    sigma = S0 / (20.0 if single else 25.0)
    for c0 in range(0, nvox, 16384):
        s = slice(c0, min(nvox, c0 + 16384))
        bb = b[None]
        if grad is None:
            dp = x[s] @ gv
        else:
            M = torch.eye(3, device=DEV)[None] + grad[s].reshape(-1, 3, 3).transpose(1, 2)
            v = M @ gv[None].expand(M.shape[0], 3, -1).contiguous()
            mag = v.norm(dim=1)
            bb = torch.where(bb > 0, bb * mag * mag, bb)
            dp = (x[s][:, :, :, None] * (v / mag[:, None]).unsqueeze(1)).sum(2)
        ds, ss = d[s, None], dstd[s, None]
        a = dp * dp
        if model == 1:
            iso, st = torch.exp(-bb * ds), torch.exp(-bb[:, None] * ds[:, None] * a)
        else:
            al, be = (ds / ss) ** 2, ss * ss / ds
            iso = torch.exp(-al * torch.log1p(bb * be))
            if model == 2:
                st = torch.exp(-al[:, None] * torch.log1p(bb[:, None] * a * be[:, None]))
            else:
                st = torch.exp(-3 * ds[:, None] / (2 * R_TRUE + 1) * bb[:, None] * ((1 - R_TRUE) * a + R_TRUE))
        m = S0[s, None] * ((1 - f[s].sum(1, keepdim=True)) * iso + (f[s][:, :, None] * st).sum(1))
        n = torch.randn(2, *m.shape, device=DEV, generator=g) * sigma[s, None]
        y[s] = torch.sqrt((m + n[0]) ** 2 + n[1] ** 2)
    return y, dict(S0=S0, d=d, dstd=dstd, f=f, x=x, sigma=sigma)


def _start_values(t, model, nf, f0, g):
    """chain starts [nvox][np] near the truth, as a fit would leave them, and tau"""
    nvox = t["S0"].numel()
    n = lambda *s: torch.randn(*s, device=DEV, generator=g)
    cols = [t["S0"] * (1 + 0.02 * n(nvox)), t["d"] * (1 + 0.05 * n(nvox))]
    if model >= 2:
        cols.append(t["dstd"] * (1 + 0.1 * n(nvox)).clamp(0.5, 1.5))
    x = t["x"] + 0.05 * n(nvox, 3, 3)
    th, ph = torch.atan2(x[..., :2].norm(dim=-1), x[..., 2]), torch.atan2(x[..., 1], x[..., 0])
    for k in range(nf):
        cols += [t["f"][:, k].clamp(min=0.01) * 0.97, th[:, k], ph[:, k]]
    if f0:
        cols.append(torch.full_like(t["S0"], 0.02))
    return torch.stack(cols, 1).cpu().numpy(), (1.0 / t["sigma"] ** 2).cpu().numpy()


def _opts(c, seed):
    o = dict(nfibres=c["nf"], model=c["model"], nburn=1000, njumps=1250, sampleevery=25, seed=seed)
    for k in ("rician", "f0"):
        if c.get(k):
            o[k] = 1
    return o


def _context(bvals, bvecs, data, opts):
    x = fdt_amd.Xfibres(**opts)
    x.set_acquisition(bvals, bvecs)
    x.load_data(data)
    return x


def _slab(c):
    """grid indices of the voxels of an ellipse in every slice"""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    X, Y = np.meshgrid(np.arange(nx), np.arange(ny))
    keep = (((X - (nx - 1) / 2) / (nx / 2)) ** 2 + ((Y - (ny - 1) / 2) / (ny / 2)) ** 2 <= 1.0).ravel()
    plane = np.nonzero(keep)[0]
    return np.concatenate([plane + nx * ny * z for z in range(nz)]).astype(np.int64)


def _net(c, seed):
    """acquisition, network weights, training rows and targets of the infer and train cases"""
    bvals, bvecs = _acquisition(c["N"], 1 if c["N"] < 70 else 3, 5)
    dims = [c["N"], 512, 512, 256, fdt_amd.SG_OUT]
    g = np.random.Generator(np.random.Philox(key=[seed, 23]))
    w = []
    for i in range(4):
        w += [g.standard_normal(dims[i] * dims[i + 1]) * math.sqrt((2.0 if i < 3 else 1.0) / dims[i]), 0.01 * g.standard_normal(dims[i + 1])]
    return bvals, bvecs, np.concatenate(w).astype(np.float32)


def _targets(t):
    """training targets [n][28] as fdt_amd.surrogate builds them, from the truth"""
    n = t["S0"].numel()
    T = torch.zeros(n, fdt_amd.SG_OUT, device=DEV)
    T[:, :3] = t["f"]
    T[:, 3:12] = t["x"].reshape(n, 9)
    T[:, 12], T[:, 13] = 1000 * t["d"], 1000 * t["dstd"]
    T[:, 14] = T[:, 17] = 1e30
    return T


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    st = dict(case=c, seed=seed)
    if kind == "queue":
        q = fdt_amd.Queue()
        for j, (N, shells, model, nf) in enumerate(QUEUE_MIX):
            bvals, bvecs = _acquisition(N, shells, seed + j)
            y, _ = _signals(bvals, bvecs, model, c["nvox"], _gen(seed, j + 1))
            q.enqueue(bvals, bvecs, y.cpu().numpy(), vox_offset=j * c["nvox"], **_opts(dict(nf=nf, model=model), seed))
        st["q"] = q
        return st
    if kind == "train":
        bvals, bvecs, w = _net(c, seed)
        y, t = _signals(bvals, bvecs, 2, c["batch"] * c["steps"], g)
        s = fdt_amd.Surrogate(c["N"], seed=1)
        s.load(w)
        T = _targets(t)
        T[:, 14:][T[:, 14:] < 1e29] = -3.0
        s.set_training_data(y.cpu().numpy(), bvals, T.cpu().numpy())
        st.update(s=s, w=w)
        return st
    if kind in ("learned", "infer"):
        if kind == "infer":
            bvals, bvecs, w = _net(c, seed)
            o = dict(nfibres=3, model=2, seed=seed)
        else:  # the acquisition that the shipped weights were trained for
            n0, shells = synth.ACQ["c1"]
            bvals, bvecs = synth.acquisition(n0, shells, synth.rng("c1", 1000))
            w = np.load(WEIGHTS)["weights"]
            o = _opts(dict(nf=3, model=2), seed)
        y, _ = _signals(bvals, bvecs, 2, c["nvox"], g)
        st["x"] = _context(bvals, bvecs, y.cpu().numpy(), o)
        s = fdt_amd.Surrogate(bvals.size, seed=1)
        s.load(w)
        st["s"] = s
        if kind == "learned":
            st["into"] = st["x"].output_buffers(alloc=fdt_amd.pinned_empty)
        return st
    bvals, bvecs = _acquisition(c["N"], c["shells"], seed)
    gidx = _slab(c) if kind == "spatial" else None
    nvox = len(gidx) if kind == "spatial" else c["nvox"]
    grad = 0.03 * torch.randn(nvox, 9, device=DEV, generator=g) if c.get("grad") else None
    y, t = _signals(bvals, bvecs, c["model"], nvox, g, grad)
    st.update(bvals=bvals, bvecs=bvecs, opts=_opts(c, seed))
    if kind == "call":
        st["data"] = y.cpu().numpy()
        return st
    st["data"] = _host(y)
    if kind == "spatial":
        st["opts"]["cpu_init"] = 1
    x = st["x"] = _context(bvals, bvecs, st["data"], st["opts"])
    if grad is not None:
        st["grad"] = grad.cpu().numpy()
    if kind == "spatial":
        st["grid"] = (c["nx"], c["ny"], c["nz"])
        st["gidx"] = gidx
    if kind == "chains":
        st["params"], st["tau"] = _start_values(t, c["model"], c["nf"], c.get("f0"), g)
    if kind != "fit":
        st["into"] = x.output_buffers(alloc=fdt_amd.pinned_empty)
    return st


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "call":
        o = dict(st["opts"])
        out = fdt_amd.run_xfibres(st["bvals"], st["bvecs"], st["data"], seed=o.pop("seed"), **o)
        del out["tau_init"]  # a Rician quantity
        return out
    if kind == "queue":
        st["q"].run()
        return [st["q"].outputs(j) for j in range(len(QUEUE_MIX))]
    if kind == "train":
        s = st["s"]
        s.load(st["w"])
        loss = [s.train_step(i * c["batch"], c["batch"], 1e-3) for i in range(c["steps"])]
        return dict(weights=s.weights(), loss=np.array(loss))
    x = st["x"]
    if kind == "infer":
        x.surrogate_start(st["s"])
        return x.get_params()[0]
    if kind == "learned":
        n = x.run_surrogate(st["s"], nburn_short=200, chi2_max=3.0, ang_max_deg=30.0)
        return dict(x.outputs(into=st["into"]), rerun=n, flags=x.fallback_flags())
    if kind == "chains":
        x.set_params(st["params"], st["tau"])
        x.mcmc()
        x.finish()
        return x.outputs(into=st["into"])
    x.load_data(st["data"])
    if "grad" in st:
        x.load_grad_dev(st["grad"])
    if kind == "fit":
        x.fit()
        return x.get_params()[:2 if c.get("rician") else 1]
    if kind == "spatial":
        x.set_grid(st["grid"], st["gidx"])
    x.run()
    return x.outputs(into=st["into"])


# ------------------------------------------------------------------ work

def _jump_flops(model, K, N, f0=False, rician=False):
    """operations of one sweep of one voxel (an FMA two, a transcendental one): every proposal's likelihood, the
    signals that the diffusivity and angle proposals change"""
    P = 3 * K + 2 + (model >= 2) + (model == 3) + bool(f0) + bool(rician)
    A, iso = {1: 3, 2: 7, 3: 5}[model], {1: 2, 2: 6, 3: 6}[model]
    R = K * A + iso + 2 * K * (6 + A)
    if model >= 2:
        R += K * A + iso if model == 2 else iso + K * A
    return N * (P * (2 * K + (33 if rician else 7)) + R)


def _chain_work(N, model, nf, nvox, jumps, f0=False, rician=False):
    scal = 2 + (model >= 2) + (model == 3) + bool(f0) + bool(rician)
    ns = 50
    out = (3 * nf + scal) * ns + scal + nf * 5
    return dict(bytes=4.0 * nvox * (N + out), flops=float(_jump_flops(model, nf, N, f0, rician)) * jumps * nvox)


def _fit_flops(N, model, nf, nvox, f0=False):
    """the LM stages at the iteration counts that its stop rule takes on such data (about 60 for the constrained
    model-1 fit, 250 over both stages of model 2 and 3)"""
    npar = 2 + 3 * nf + (model >= 2) + bool(f0)
    return float(N * (npar * (npar + 1) + 2 * npar + 40 * nf)) * (60 if model == 1 else 250) * nvox


def work(case):
    c = case
    kind = c["kind"]
    if kind == "queue":
        both = [_chain_work(N, m, k, c["nvox"], 2250) for N, _, m, k in QUEUE_MIX]
        fl = sum(w["flops"] for w in both) + sum(_fit_flops(N, m, k, c["nvox"]) for N, _, m, k in QUEUE_MIX)
        return dict(bytes=sum(w["bytes"] for w in both), flops=fl)
    if kind == "learned":
        w = _chain_work(288, 2, 3, c["nvox"], 1450)
        return dict(bytes=w["bytes"], flops=w["flops"] + 2.0 * c["nvox"] * (288 * 512 + 512 * 512 + 512 * 256 + 256 * 28))
    if kind == "infer":
        per = c["N"] * 512 + 512 * 512 + 512 * 256 + 256 * 28
        return dict(bytes=4.0 * c["nvox"] * (c["N"] + 28) + 2.0 * per, flops=2.0 * per * c["nvox"])
    if kind == "train":
        per = c["N"] * 512 + 512 * 512 + 512 * 256 + 256 * 28
        rows = c["batch"] * c["steps"]
        return dict(bytes=2.0 * rows * c["N"] + 4.0 * rows * 28 + 30.0 * per * c["steps"], flops=6.0 * per * rows)
    nvox = len(_slab(c)) if kind == "spatial" else c["nvox"]
    if kind == "fit":
        npar = 2 + 3 * c["nf"] + (c["model"] >= 2) + bool(c.get("f0"))
        return dict(bytes=4.0 * nvox * (c["N"] + npar), flops=_fit_flops(c["N"], c["model"], c["nf"], nvox, c.get("f0")))
    w = _chain_work(c["N"], c["model"], c["nf"], nvox, 2250, c.get("f0"), c.get("rician"))
    if kind in ("call", "run"):
        w["flops"] += _fit_flops(c["N"], c["model"], c["nf"], nvox, c.get("f0"))
    return w


# ------------------------------------------------------------------ exact

def _layers(w, n_in):
    dims, out, o = [n_in, 512, 512, 256, fdt_amd.SG_OUT], [], 0
    for i in range(4):
        n = dims[i] * dims[i + 1]
        out += [w[o:o + n].reshape(dims[i], dims[i + 1]), w[o + n:o + n + dims[i + 1]]]
        o += n + dims[i + 1]
    return out


def _forward(p, X):
    for i in range(4):
        X = X @ p[2 * i] + p[2 * i + 1]
        if i < 3:
            X = torch.nn.functional.gelu(X)
    return X


def _normalised(y, bvals):
    b0 = torch.tensor(bvals <= 50.0, device=DEV)
    y = y.double()
    s0 = y[:, b0].mean(1)
    return y / s0[:, None], s0


def exact(case, seed):
    """the network's outputs in 64 bits.  A chain has no such value: it is one realisation of a random sequence of
    accept/reject decisions, and another rounding gives another one of the same posterior.  Nor has a fit: the
    Levenberg loop ends where its relative-cost test ends it, on flat directions well before a minimum."""
    c = case
    if c["kind"] == "infer":
        bvals, bvecs, w = _net(c, seed)
        y, _ = _signals(bvals, bvecs, 2, c["nvox"], _gen(seed))
        p = _layers(torch.tensor(w, device=DEV).double(), c["N"])
        out = []
        for c0 in range(0, c["nvox"], 32768):
            X, s0 = _normalised(y[c0:c0 + 32768], bvals)
            o = _forward(p, X)
            f = o[:, :3].clamp(0.01, 0.95)
            fs = f.sum(1, keepdim=True)
            f = torch.where(fs > 0.95, f * (0.95 / fs), f)
            v = o[:, 3:12].reshape(-1, 3, 3)
            th, ph = torch.atan2(v[..., :2].norm(dim=-1), v[..., 2]), torch.atan2(v[..., 1], v[..., 0])
            cols = [s0, (o[:, 12] * 1e-3).clamp(1e-5, 0.0049), (o[:, 13] * 1e-3).clamp(1e-5, 0.0099)]
            for k in range(3):
                cols += [f[:, k], th[:, k], ph[:, k]]
            out.append(torch.stack(cols, 1))
        return torch.cat(out).cpu().numpy()
    if c["kind"] == "train":
        bvals, bvecs, w = _net(c, seed)
        y, t = _signals(bvals, bvecs, 2, c["batch"] * c["steps"], _gen(seed))
        X, _ = _normalised(y, bvals)
        T = _targets(t).double()
        T[:, 14:][T[:, 14:] < 1e29] = -3.0
        used = (T < 1e29).double()
        flat = torch.tensor(w, device=DEV).double()
        m, v, losses = torch.zeros_like(flat), torch.zeros_like(flat), []
        for i in range(c["steps"]):
            r = slice(i * c["batch"], (i + 1) * c["batch"])
            q = flat.clone().requires_grad_(True)
            o, tt = _forward(_layers(q, c["N"]), X[r]), T[r]
            pr, x = o[:, 3:12].reshape(-1, 3, 3), tt[:, 3:12].reshape(-1, 3, 3)
            pp = (pr * pr).sum(2)
            loss = ((o[:, :3] - tt[:, :3]) ** 2).sum() + ((o[:, 12:14] - tt[:, 12:14]) ** 2).sum()
            loss = loss + (tt[:, :3].clamp(min=0) * (pp * pp - 2 * (pr * x).sum(2) ** 2 + 1)).sum()
            loss = loss + 0.1 * (used[r, 14:] * (o[:, 14:] - tt[:, 14:] * used[r, 14:]) ** 2).sum()
            loss = loss / c["batch"]
            loss.backward()
            losses.append(float(loss))
            m = 0.9 * m + 0.1 * q.grad
            v = 0.999 * v + 0.001 * q.grad ** 2
            flat = flat - 1e-3 * (m / (1 - 0.9 ** (i + 1))) / ((v / (1 - 0.999 ** (i + 1))).sqrt() + 1e-8)
        return dict(weights=flat.cpu().numpy(), loss=np.array(losses))
    return None
