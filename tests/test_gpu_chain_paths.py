"""Every chain kernel that a launch can take gives the same chains: an
acquisition that fills its tile (no padding masks) and the same one in the next
larger tile (masked), with one row and with two rows per voxel."""
import numpy as np
import pytest

from fdt_amd import synth
from test_gpu_launch_sizes import starts

pytestmark = pytest.mark.gpu


def volume(n, nvox, model, b0, seed=1, snr=25.0):
    """nvox voxels of `model` on an n-volume acquisition with b0 volumes of b = 0 and three shells: acquisition, data and
    the truth behind them"""
    g = np.random.Generator(np.random.Philox(key=[seed, n]))
    bvals, bvecs = synth.acquisition(b0, [(1000.0 * (i + 1), (n - b0) // 3 + (i < (n - b0) % 3)) for i in range(3)], g)
    S0, d = g.uniform(800, 1200, nvox), g.uniform(1e-3, 2e-3, nvox)
    dstd = d * g.uniform(0.1, 0.5, nvox)
    f = g.dirichlet(np.ones(3), nvox) * g.uniform(0.3, 0.8, nvox)[:, None]
    x = synth.unit_vectors(g, 3 * nvox).reshape(nvox, 3, 3)
    sig = synth.clean_signal(model, bvals, bvecs, S0, d, dstd, f, x)
    sd = (S0 / snr)[:, None]
    data = np.hypot(sig + sd * g.standard_normal(sig.shape), sd * g.standard_normal(sig.shape)).astype(np.float32)
    th, ph = np.arccos(x[..., 2]), np.arctan2(x[..., 1], x[..., 0])
    return (bvals, bvecs), data, dict(S0=S0, d=d, dstd=dstd, f=f, th=th, ph=ph, tau=1 / sd[:, 0] ** 2)


def chain_starts(t, model, K, opts):
    p = starts(t, model, K)
    if opts.get("f0"):
        p = np.concatenate([p, np.full((len(p), 1), 0.03, np.float32)], 1)
    return p, t["tau"].astype(np.float32)


def run(fdt, acq, data, params, tau, tile=0, **opts):
    """chains of `data` from given starts: everything that a caller can read"""
    x = fdt.Xfibres(**dict(dict(nburn=20, njumps=40, sampleevery=10, updateproposalevery=15), **opts))
    try:
        x.set_mcmc_tile(tile)
        x.set_acquisition(*acq)
        x.load_data(data)
        x.set_params(params, tau)
        x.mcmc(7)
        x.finish()
        return dict(x.outputs(), widths=x.widths().T, energy=x.energy())
    finally:
        x.close()


def repeat(a, n):
    return np.tile(a, (-(-n // len(a)),) + (1,) * (a.ndim - 1))[:n]


def assert_same(a, b, n, what):
    for k in a:
        np.testing.assert_array_equal(a[k][..., :n], b[k][..., :n], err_msg=f"{what}: {k}")


# 24 voxels run in two rows from 113 volumes on, 4,201 in one row up to 288 volumes (one fibre: 448)
@pytest.mark.parametrize("nvox", [24, 4201])
@pytest.mark.parametrize("n,larger,model,K,opts", [
    (48, 5, 1, 2, {}), (48, 5, 2, 3, dict(rician=1)), (80, 7, 2, 2, dict(f0=1)), (80, 7, 3, 1, dict(rician=1)),
    (112, 10, 3, 3, {}), (112, 10, 1, 1, dict(rician=1, f0=1, ardf0=1)), (160, 14, 2, 3, dict(f0=1, ardf0=1)),
    (160, 14, 2, 2, dict(rician=1)), (224, 18, 1, 3, dict(all_ard=1)), (224, 18, 3, 3, dict(rician=1)),
    (288, 24, 2, 1, {}), (384, 28, 2, 3, {}), (384, 28, 1, 1, {}), (384, 28, 3, 2, dict(rician=1)),
    (448, 32, 3, 2, dict(f0=1)), (448, 32, 2, 3, dict(rician=1, no_ard=1))])
def test_filled_tiles_match_the_next_larger_one(fdt, n, larger, model, K, opts, nvox):
    acq, data, t = volume(n, 24, model, b0=min(n // 16, 12))  # below 16: no slot of b = 0 volumes, one order in every tile
    p, tau = chain_starts(t, model, K, opts)
    opts = dict(opts, nfibres=K, model=model)
    args = (fdt, acq, repeat(data, nvox), repeat(p, nvox), repeat(tau, nvox))
    assert_same(run(*args, **opts), run(*args, tile=larger, **opts), nvox, f"N={n} model {model} K={K} {opts}")


@pytest.mark.parametrize("n,nvox,K,rician,lanes,vpl", [
    (69, 100, 2, 0, 16, 5), (112, 100, 1, 1, 16, 7), (113, 2048, 2, 0, 32, 5), (160, 2049, 2, 0, 16, 10),
    (200, 4096, 1, 1, 32, 7), (200, 4097, 1, 1, 16, 14), (288, 2049, 3, 0, 16, 18), (289, 3000, 2, 0, 32, 12),
    (289, 3000, 1, 0, 16, 24), (448, 5000, 1, 1, 32, 14), (512, 3000, 1, 0, 32, 16)])
def test_timing_reports_the_lanes_of_a_voxel(fdt, n, nvox, K, rician, lanes, vpl):
    """fdt_timing: volumes per lane and lanes per voxel, of which their product holds the acquisition"""
    acq, data, t = volume(n, 24, 1, b0=4)
    x = fdt.Xfibres(nfibres=K, model=1, rician=rician, nburn=0, njumps=2, sampleevery=1)
    try:
        x.set_acquisition(*acq)
        x.load_data(repeat(data, nvox))
        x.set_params(repeat(starts(t, 1, K), nvox), repeat(t["tau"].astype(np.float32), nvox))
        x.mcmc(0)
        tm = x.timing()
        assert (tm["lanes"], tm["vpl"]) == (lanes, vpl)
        x.set_mcmc_tile(32)
        x.mcmc(0)
        tm = x.timing()
        assert tm["lanes"] * tm["vpl"] == 512
    finally:
        x.close()
