"""LM fits with a row of 16 lanes and with a whole wave per voxel (the kernel of
large and of small launches) are equal to the last bit: beyond one step of 64
volumes and at its edges, with and without a b-shell table, with --gradnonlin
and --f0, in the three precision modes.  The kernel of large launches also
follows the oracle by itself."""
import numpy as np
import pytest

from fdt_amd import synth
from test_gpu_chain_paths import repeat, volume

pytestmark = pytest.mark.gpu

FEW, MANY = 29, 17021  # a wave per voxel; a row per voxel in every mode and on every kernel's occupancy


def fit(fdt, acq, data, grad=None, **opts):
    x = fdt.Xfibres(**opts)
    try:
        x.set_acquisition(*acq)
        x.load_data(data)
        if grad is not None:
            x.load_grad_dev(grad)
        x.fit()
        p, tau = x.get_params()
        return p, x.lm_iters(), tau
    finally:
        x.close()


def jittered(acq, seed=5):
    """more than 16 distinct b values: no shell table"""
    bvals, bvecs = acq
    g = np.random.default_rng(seed)
    return np.where(bvals > 0, bvals + g.uniform(-30, 30, bvals.shape), 0).astype(np.float32), bvecs


@pytest.mark.parametrize("n,model,K,opts,shells,gn", [
    (64, 1, 2, {}, True, False), (65, 2, 3, {}, True, False), (128, 2, 1, {}, True, False),
    (145, 1, 1, dict(f0=1), True, False), (145, 2, 2, {}, True, True), (145, 2, 3, {}, False, False),
    (69, 1, 3, dict(lm_fp64=1), True, False), (69, 3, 1, dict(lm_fp64=1), True, False),
    (69, 1, 1, dict(nonlin=1), True, False), (69, 2, 2, {}, True, False), (69, 3, 3, {}, False, True),
    (288, 2, 3, {}, True, False), (288, 3, 2, {}, True, False), (288, 1, 3, dict(nonlin=1), False, False),
    (288, 2, 3, dict(lm_fp64=0), True, False), (288, 2, 1, dict(f0=1), True, False),
    (193, 2, 3, dict(f0=1), False, False), (432, 2, 2, dict(rician=1), True, False)])
def test_a_row_and_a_wave_per_voxel(fdt, n, model, K, opts, shells, gn):
    acq, data, _ = volume(n, FEW, model, b0=max(2, n // 16))
    if not shells:
        acq = jittered(acq)
    grad = synth.grad_dev(np.random.default_rng(n), FEW) if gn else None
    opts = dict(opts, nfibres=K, model=model)
    a = fit(fdt, acq, data, grad, **opts)
    b = fit(fdt, acq, repeat(data, MANY), None if grad is None else repeat(grad, MANY), **opts)
    assert np.isfinite(a[0]).all()
    for k, u, v in zip(("parameters", "iterations", "tau"), a, b):
        if k != "tau" or opts.get("rician"):
            np.testing.assert_array_equal(u, v[:FEW], err_msg=k)


@pytest.mark.parametrize("name,model,K,opts", [("c0", 1, 2, {}), ("c1", 2, 3, {}), ("c1", 3, 2, {}), ("c1", 2, 2, dict(f0=1))])
def test_a_row_per_voxel_matches_oracle(orc, fdt, name, model, K, opts):
    """a launch of 17,021 voxels (384 different ones, repeated) in FP64, at the bar of the pipeline tests: within 1e-4
    of the oracle on as many voxels as the oracle on data perturbed by 1e-8, less three standard deviations"""
    from test_gpu_lm import lm_errors
    nvox = 384
    v = synth.voxels(name, nvox)
    y = v["data"].astype(np.float64)
    o = orc.opts(nfibres=K, model=model, **opts)
    want, _, _ = orc.fit(o, v["bvals"], v["bvecs"], y)
    near, _, _ = orc.fit(o, v["bvals"], v["bvecs"], y * (1 + 1e-8 * np.random.default_rng(1).standard_normal(y.shape)))
    got = fit(fdt, (v["bvals"], v["bvecs"]), repeat(v["data"], MANY), nfibres=K, model=model, lm_fp64=1, **opts)[0]
    kind, f0 = 2 if model >= 2 else 1, bool(opts.get("f0"))
    within = np.mean(lm_errors(got[:nvox].astype(np.float64), want, kind, K, f0) < 1e-4)
    floor = np.mean(lm_errors(near, want, kind, K, f0) < 1e-4)
    print(f"{name} model {model} K={K} {opts}: within 1e-4 of the oracle on {within:.3f} of voxels (floor {floor:.3f})")
    assert within >= floor - 3 * np.sqrt(max(floor * (1 - floor), 0.01) / nvox)
    np.testing.assert_array_equal(got, repeat(got[:nvox], MANY))
