"""Kernels that are chosen by the size of a launch give the same results as
the ones beside them: chains with one and two rows per voxel, LM fits with a
row and with a whole wave per voxel, the network's product in its tiles.  Each
test runs a few voxels alone and as the first of a launch large enough for the
other kernel; results are equal to the last bit, as every sum is taken in the
same order.  Rician chains at low signal, where both series of log I0 occur in
one wave, follow the oracle draw for draw."""
import numpy as np
import pytest

from fdt_amd import synth

pytestmark = pytest.mark.gpu


def volume(n, nvox, model, seed=1, snr=25.0):
    """nvox voxels of model `model` on an n-volume acquisition (one b = 0 volume in 16), and chain starts near the truth"""
    g = np.random.Generator(np.random.Philox(key=[seed, n]))
    n0 = max(2, n // 16)
    dirs = [(n - n0) // 3 + (1 if i < (n - n0) % 3 else 0) for i in range(3)]
    bvals, bvecs = synth.acquisition(n0, [(1000.0 * (i + 1), m) for i, m in enumerate(dirs)], g)
    S0, d = g.uniform(800, 1200, nvox), g.uniform(1e-3, 2e-3, nvox)
    dstd = d * g.uniform(0.1, 0.5, nvox)
    f = g.dirichlet(np.ones(3), nvox) * g.uniform(0.3, 0.8, nvox)[:, None]
    x = synth.unit_vectors(g, 3 * nvox).reshape(nvox, 3, 3)
    sig = synth.clean_signal(model, bvals, bvecs, S0, d, dstd, f, x)
    sd = (S0 / snr)[:, None]
    data = np.hypot(sig + sd * g.standard_normal(sig.shape), sd * g.standard_normal(sig.shape)).astype(np.float32)
    th, ph = np.arccos(x[..., 2]), np.arctan2(x[..., 1], x[..., 0])
    return bvals, bvecs, data, dict(S0=S0, d=d, dstd=dstd, f=f, th=th, ph=ph, tau=1 / sd[:, 0] ** 2)


def starts(t, model, K):
    cols = [t["S0"], t["d"]] + ([t["dstd"]] if model >= 2 else [])
    for k in range(K):
        cols += [t["f"][:, k], t["th"][:, k], t["ph"][:, k]]
    return np.stack(cols, 1).astype(np.float32)


def chains(fdt, bvals, bvecs, data, params, tau, **opts):
    x = fdt.Xfibres(nburn=20, njumps=40, sampleevery=10, updateproposalevery=15, **opts)
    try:
        x.set_acquisition(bvals, bvecs)
        x.load_data(data)
        x.set_params(params, tau)
        x.mcmc(7)
        x.finish()
        return dict(x.outputs(), widths=x.widths().T, energy=x.energy())
    finally:
        x.close()


# the edges of the tiles with two rows (10, 14, 18, 24, 28 and 32 volumes in 16 lanes), each model and fibre count
@pytest.mark.parametrize("n,model,K,rician", [
    (113, 1, 1, 0), (160, 2, 3, 0), (161, 3, 2, 0), (224, 2, 2, 0), (225, 1, 3, 0), (288, 2, 3, 0), (288, 3, 1, 0),
    (289, 2, 1, 0), (385, 1, 1, 0), (448, 3, 1, 0),
    (144, 1, 2, 1), (200, 2, 1, 1), (257, 2, 3, 1), (288, 3, 3, 1)])
def test_chains_in_one_and_two_rows(fdt, n, model, K, rician):
    few, many = 24, 4112
    bvals, bvecs, data, t = volume(n, few, model)
    p, tau = starts(t, model, K), t["tau"].astype(np.float32)
    opts = dict(nfibres=K, model=model, rician=rician)
    rep = (many + few - 1) // few
    a = chains(fdt, bvals, bvecs, data, p, tau, **opts)
    b = chains(fdt, bvals, bvecs, np.tile(data, (rep, 1))[:many], np.tile(p, (rep, 1))[:many], np.tile(tau, rep)[:many], **opts)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k][..., :few], err_msg=f"N={n} model {model} K={K}: {k}")


@pytest.mark.parametrize("model,K,opts", [
    (1, 1, {}), (1, 2, dict(nonlin=1)), (1, 3, {}), (2, 2, {}), (2, 3, {}), (3, 3, {}), (2, 3, dict(lm_fp64=1)),
    (2, 2, dict(lm_fp64=0)), (2, 2, dict(f0=1)), (2, 2, dict(rician=1))])
@pytest.mark.parametrize("n", [20, 33])
def test_fits_with_a_row_and_a_wave_per_voxel(fdt, n, model, K, opts):
    few, many = 29, 17000
    bvals, bvecs, data, _ = volume(n, few, model)
    out = []
    for d in (data, np.tile(data, ((many + few - 1) // few, 1))[:many]):
        x = fdt.Xfibres(nfibres=K, model=model, **opts)
        try:
            x.set_acquisition(bvals, bvecs)
            x.load_data(d)
            x.fit()
            p, tau = x.get_params()
            out.append((p[:few], x.lm_iters()[:few], tau[:few] if "rician" in opts else None))
        finally:
            x.close()
    for a, b in zip(*out):
        if a is not None:
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n_in", [33, 72, 288])
def test_network_in_its_tiles(fdt, n_in):
    g = np.random.default_rng(n_in)
    x = g.uniform(50, 1000, (9001, n_in)).astype(np.float32)
    b = np.where(np.arange(n_in) < 5, 0.0, 1000.0)
    s = fdt.Surrogate(n_in, seed=3)
    try:
        whole = s.forward(x, b)
        for n in (1, 31, 33, 300, 4097):
            np.testing.assert_array_equal(s.forward(x[:n], b), whole[:n], err_msg=f"{n} rows")
    finally:
        s.close()


@pytest.mark.parametrize("n,K", [(60, 1), (100, 2), (288, 3)])
def test_rician_chains_at_low_signal_track_oracle(orc, fdt, n, K):
    """SNR 4: tau p y runs from below 1 to 30, so waves meet log I0 on both sides of 3.75; the bar of the other
    draw-for-draw tests"""
    bvals, bvecs, data, t = volume(n, 48, 2, snr=4.0)
    p, tau = starts(t, 2, K), t["tau"].astype(np.float32)
    run = dict(nfibres=K, model=2, rician=1, nburn=0, njumps=50, sampleevery=25)
    x = fdt.Xfibres(**run)
    try:
        x.set_acquisition(bvals, bvecs)
        x.load_data(data)
        x.set_params(p, tau)
        x.mcmc(0)
        x.finish()
        got = x.outputs()
    finally:
        x.close()
    o = orc.mcmc(orc.opts(**run), bvals, bvecs, data.astype(np.float64), p.astype(np.float64), tau.astype(np.float64))
    orc.finish(orc.opts(**run), o)
    same = np.all(np.abs(got["f"][:, 0, :] - o["f"][:, 0, :]) < 1e-3, axis=0) & (np.abs(got["d"][0] / o["d"][0] - 1) < 1e-3)
    print(f"N={n} K={K}: first sample agrees on {same.mean():.3f} of voxels")
    assert same.mean() >= 0.75
