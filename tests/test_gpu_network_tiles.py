"""The network's gradients at batches large enough for the wide tiles of its
products (the bar of the 257-row gradient test), and the weight gradients at row
counts that end inside a K step."""
import numpy as np
import pytest

from fdt_amd import synth
from oracle import mlp_oracle as M
from test_gpu_chain_paths import repeat
from test_gpu_surrogate import rand_targets, rel

pytestmark = pytest.mark.gpu


# 64 x 64 tiles of dZ.W^T from 2,017 rows (512 columns), 128 x 128 from 8,065; 32 x 32 below
@pytest.mark.parametrize("name,batch", [("c0", 33), ("c0", 2050), ("c1", 8100)])
def test_gradients_match_oracle_in_every_tile(fdt, name, batch):
    v = synth.voxels(name, 512)
    data = repeat(v["data"], batch)
    t = rand_targets(np.random.default_rng(batch), batch)
    s = fdt.Surrogate(v["bvals"].size, seed=5)
    try:
        layers = [(W.astype(np.float64), b.astype(np.float64)) for W, b in s.layers()]
        s.set_training_data(data, v["bvals"], t)
        gg, loss = s.gradients(0, batch)
        go, loss_o = M.backward(M.normalise(data, v["bvals"]), layers, t, emulate_bf16=True)
        assert loss == pytest.approx(loss_o, rel=1e-2)
        for l, (W, b) in enumerate(s.layers(gg)):
            eW, eb = rel(W, go[l][0]), rel(b, go[l][1])
            print(f"{name}, {batch} rows, layer {l}: dW rel err {eW:.2e}, db rel err {eb:.2e}")
            assert eW < 3e-2 and eb < 3e-2
    finally:
        s.close()
